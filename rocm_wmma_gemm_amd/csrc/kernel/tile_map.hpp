// Workgroup id -> output tile, for a chip whose 256 CUs sit in 8 XCDs with one
// L2 each.  The hardware deals consecutive workgroup ids round-robin over the
// XCDs, so ids that are congruent mod 8 share an L2.  The map first renumbers
// the ids so that every XCD owns one contiguous run of "logical" ids, then walks
// the tile grid in bands of `group` tile rows (or columns), column by column inside a band,
// so that a run of logical ids covers a compact group x (run/group) rectangle of
// C and re-uses the same A row panels and B column panels out of that L2.
//
// Plays the role of the reference's tile_mapper (reference
// rocm_wmma_gemm/include/rocm_wmma_gemm/kernel/mapping.hpp:34-324); unlike the
// reference's maps it is a bijection for every grid, with no clamping.
#ifndef ROCM_WMMA_GEMM_TILE_MAP_HPP
#define ROCM_WMMA_GEMM_TILE_MAP_HPP

#if defined(__HIPCC__)
#define RWG_HD __host__ __device__
#else
#define RWG_HD
#endif

namespace rocm_wmma_gemm
{
namespace device
{

constexpr int num_xcd = 8;

struct tile_coord
{
    int m;
    int n;
};

// Contiguous-per-XCD renumbering of [0, total).
RWG_HD inline int xcd_remap(int wg, int total)
{
    const int per_xcd = (total + num_xcd - 1) / num_xcd; // ids owned by a "tall" XCD
    const int rem     = total % num_xcd;
    const int tall    = rem == 0 ? num_xcd : rem; // XCDs that own per_xcd ids
    const int xcd     = wg % num_xcd;
    const int local   = wg / num_xcd;
    if(xcd < tall)
    {
        return xcd * per_xcd + local;
    }
    return tall * per_xcd + (xcd - tall) * (per_xcd - 1) + local;
}

// Banded walk.  group > 0: bands of `group` tile rows; inside a band, down a column
// first.  group < 0: the mirror image, bands of -group tile columns, along a row first
// (a grid that is wider than tall then gives an XCD the rectangle that the upright walk
// gives it on the transposed grid).  group 0 counts as 1.
RWG_HD inline tile_coord banded_tile(int id, int grid_m, int grid_n, int group)
{
    const bool mirrored = group < 0;
    const int  g        = mirrored ? -group : (group == 0 ? 1 : group);
    const int  tall     = mirrored ? grid_n : grid_m; // the dimension the bands cut
    const int  wide     = mirrored ? grid_m : grid_n;
    const int  per_band = g * wide;
    const int  band     = id / per_band;
    const int  first    = band * g;
    const int  rows     = (tall - first) < g ? (tall - first) : g;
    const int  in_band  = id - band * per_band;
    const int  along    = first + in_band % rows;
    const int  across   = in_band / rows;
    tile_coord t;
    t.m = mirrored ? across : along;
    t.n = mirrored ? along : across;
    return t;
}

RWG_HD inline tile_coord map_tile(int wg, int grid_m, int grid_n, int group)
{
    return banded_tile(xcd_remap(wg, grid_m * grid_n), grid_m, grid_n, group);
}

// What one workgroup works on.  Ids enumerate the whole tiles first, then (slice, split
// tile) pairs, slices outermost.
struct block_work
{
    int  tile_id; // position in the tile walk
    int  slice, slices; // K slice of this workgroup and how many the tile has (1 = whole K)
    bool walk_order; // tile_id counts along the walk already (see tile_of), else it is dealt by XCD
};

// Where every tile is split, the ids of the launch are renumbered as a whole, so that an XCD
// owns a contiguous run of (slice, tile) pairs, a slice or two of K over all tiles.  Its L2 then
// fetches its part of A and B once, instead of nearly all of both as with the tiles of every
// slice dealt over the XCDs like whole tiles.  What the eight L2s fetch in a launch: 704 x 896 x 12096 in 16
// slices 147 -> 62 MB (the operands are 39), the call 47.7 -> 44.5 us; 2048 x 1024 x 32768 in 8,
// 538 -> 438 MB of 201, 145.7 -> 137.3 us (operands from HBM).  A few slices of many tiles gain nothing and
// lose nothing.
RWG_HD inline block_work decode_block(int b, int tiles, int tail_begin, int k_slices)
{
    if(b < tail_begin || k_slices == 1)
    {
        return {b, 0, 1, false};
    }
    const int split_tiles = tiles - tail_begin;
    if(tail_begin == 0)
    {
        const int item  = xcd_remap(b, split_tiles * k_slices);
        const int slice = item / split_tiles;
        return {item - slice * split_tiles, slice, k_slices, true};
    }
    const int r     = b - tail_begin;
    const int slice = r / split_tiles;
    return {tail_begin + (r - slice * split_tiles), slice, k_slices, false};
}

RWG_HD inline tile_coord tile_of(const block_work& w, int grid_m, int grid_n, int group)
{
    return banded_tile(w.walk_order ? w.tile_id : xcd_remap(w.tile_id, grid_m * grid_n), grid_m, grid_n, group);
}

} // namespace device
} // namespace rocm_wmma_gemm

#endif // ROCM_WMMA_GEMM_TILE_MAP_HPP
