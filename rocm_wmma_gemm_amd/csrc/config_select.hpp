// Shape -> launch plan.  The tuned table comes from gemm_config_gfx950_*.json via
// config/generate_config.py; shapes the table does not name are served by a time
// estimate over the compiled variants (select_plan says which), skinny ones with unaligned rows by
// the general kernel, the rest by the table's nearest entry, and layouts the
// table does not cover at all by a shape heuristic.
//
// select_plan_from follows the reference's generated find_best_config /
// find_closest_config (reference rocm_wmma_gemm/config/generate_config.py:174-271):
//   1. exact (M, N, K, type group, layouts) hit;
//   2. for the fp32-output group, an exact hit in the 16-bit-output group;
//   3. nearest entry with the same type group and layouts: nearest K first, then
//      smallest squared (M, N) distance; an empty group falls back to group 0.
// Unlike the reference there is no sentinel index doubling as "not found", so a
// genuine hit on any entry is honoured.
#ifndef ROCM_WMMA_GEMM_CONFIG_SELECT_HPP
#define ROCM_WMMA_GEMM_CONFIG_SELECT_HPP

#include <cstddef>

namespace rocm_wmma_gemm
{
namespace host
{

struct launch_plan
{
    int variant; // index into the compiled variant table
    int swizzle; // band height of the tile map: s > 0 bands of s tile rows, s < 0 bands of -s tile columns
    int split_k; // K slices (1 = off); -s (s > 1) = split only the last, partial wave of tiles s
                 // ways; -1 = persistent kernel walks by K tile (equal K tiles per workgroup)
    int touch = 0; // persistent kernel, two small fields.  Bits 0-3: d > 0 = touch the cache lines of
                   // the K tile d tiles past the one being loaded (see gemm_args::warm_ahead); 0 = off.
                   // Bits 4-7: c > 0 = walk the K tiles in runs of 2^(c-1), the XCDs out of step by
                   // whole runs (see gemm_args::k_block); 0 = in order.
                   // Bits 8-9: c > 0 = within groups of 2^c K tiles the workgroups start at different
                   // tiles (see gemm_args::k_group); 0 = in order.
};

// the two fields of launch_plan::touch
constexpr int plan_touch_distance(int touch)
{
    return touch & 15;
}
constexpr int plan_k_run(int touch)
{
    return ((touch >> 4) & 15) == 0 ? 0 : 1 << (((touch >> 4) & 15) - 1);
}
constexpr int plan_k_group(int touch)
{
    return ((touch >> 8) & 3) == 0 ? 0 : 1 << ((touch >> 8) & 3);
}
// run: 0 or a power of two up to 16; group: 0, 2, 4 or 8
constexpr int plan_touch_field(int distance, int run, int group = 0)
{
    int code = 0;
    for(int r = run; r > 0; r >>= 1)
    {
        ++code;
    }
    return (distance & 15) | (code << 4) | ((group == 2 ? 1 : group == 4 ? 2 : group == 8 ? 3 : 0) << 8);
}

struct tuned_entry
{
    size_t m, n, k;
    int    type_group; // 0: C is 16-bit (f16_f16, bf16_bf16); 1: C is fp32
    int    layout_a, layout_b, layout_c; // 0 row-major, 1 column-major
    launch_plan plan;
};

// Constants of model_plan's time estimate (microseconds, bytes per microsecond), measured
// on the GPU: config/fit_model.py fits them to a tuner log, config/model_<arch>.json keeps
// them and config/generate_config.py copies them into the generated header.
struct model_step
{
    int    pipeline, block_m, block_n;
    double step_us; // per K tile of 64 with every compute unit at work
    double item_us; // per tile: the stores of C and the turn to the next tile
};
// Constants of the estimate for the plans of the whole-K streaming kernel (pipeline 7),
// fitted by config/fit_model.py --stream to a sweep of config/sweep_stream.py.
struct model_stream
{
    double launch_us, fill_us; // per launch; per pass over the compute units (the ring fills)
    double exchange_us; // several workgroups per tile: the partial tiles through memory ...
    double exchange_us_per_kb; // ... and per KiB of them that the last workgroup adds up
    double bytes_per_us_kmajor, bytes_per_us_other; // stream of the large operand from memory
    double bytes_per_us_l2; // the small operand, which every workgroup reads from L2
    double transposed_operand; // relative cost of a stage per operand that is not K-contiguous
    double panel_sharing; // how much of a panel of the large operand that g workgroups read
                          // is fetched once for all: it counts as fetched g / (1 + (g - 1) x this) times
    double half_line; // factor on a rate for an operand contiguous along M or N on a 32-wide side
                      // of the tile: requests of 64 bytes, half a cache line
    double beyond_cache, beyond_cache_other; // factors on the two rates from memory for a large
                         // operand over 256 MB, K-contiguous or not (set by hand, not fitted)
    double taking_turns; // two workgroups on a compute unit: a stage of each takes 1 + this of what
                         // it takes alone, where the compute unit is the bound (set by hand)
    double stage_us[8]; // per stage of 128 of one compute unit: tiles 32x32, 64x32, 32x64, 64x64,
                        // 16x32, 16x64, 32x16, 64x16
};
struct model_constants
{
    int    compute_units; // of the GPU the constants were measured on
    double launch_us, reduce_us;
    double plane_bytes_per_us; // split-K partial planes: written, then read by the reduce kernel
    double tile_bytes_per_us; // partial tiles of a split tail wave or of the walk by K tile
    double copy_bytes_per_us; // padded operand copies
    double operand_bytes_per_us; // what the tiled kernels reach at most streaming A and B from memory
                                 // (skinny shapes: 134 MB in 24-27 us of split-K kernel, 470 MB in 83-96; set by hand)
    const model_step* steps;
    int               step_count;
    model_stream      stream;
};
extern const model_constants model_measured;

// Defined in config_select.cpp
extern const tuned_entry* const tuned_table;
extern const size_t             tuned_count;

// Pure functions over a table (unit-testable with any table).
bool find_exact(const tuned_entry* table, size_t count, size_t m, size_t n, size_t k,
                int type_group, int la, int lb, int lc, launch_plan* out);
bool find_closest(const tuned_entry* table, size_t count, size_t m, size_t n, size_t k,
                  int type_group, int la, int lb, int lc, launch_plan* out);
launch_plan heuristic_plan(size_t m, size_t n, size_t k, int lc);
// Operations per element copied from which on padded copies pay against the general kernel: 256, and
// 200 where its way of loading costs more.  Unaligned rows, which it reads a few bytes at a time, from a K of
// 256 on: about 100 rows against an odd weight (64 x 4096 x 4095: 32.8 us copied, 20.5 by the general kernel; 96
// rows 33.7 and 27.4; 133 x 5000 x 3001 43.1 and 278; 441 x 806 x 150 13.4 and 9.9).  Aligned rows from a K
// of 2048 and 5120 columns on (133 x 5560 x 10232, 251 of them, 89 us copied, 133 by the next best plan, 131 x
// 11920 x 2696 0.64 of its time; with fewer columns, 133 x 1088 x 4672 26 and 17; 832 x 128 x 128, 238 of them, 12.4
// copied and 6.0 by the general kernel's 128 x 128 tile).
constexpr double copy_pays_flops_aligned = 256.0, copy_pays_flops = 200.0;

// The padded copies that a direct-to-LDS tile needs of the operands of one problem, in kernel
// space: what the launch makes of them and what the estimate prices.
struct operand_copies
{
    bool   a, b; // which operands are copied ...
    size_t lda, ldb; // ... their leading dimensions, copied or not ...
    size_t elems_a, elems_b; // ... and the elements of a copy, per batch entry (0: none)
    bool   pays; // there is something to copy and the GEMM is large next to it
};
// a_rows, b_rows: the operand's rows start on 16 bytes.  edges: the tile's kernel cuts ragged edges off
// itself (the persistent one), so that only an operand whose rows are not aligned is copied, its
// rows padded (a K-contiguous one's to whole K tiles) and their number left as it is; every other
// kernel needs whole tiles.
operand_copies padded_copies(size_t m, size_t n, size_t k, bool a_kmajor, bool b_kmajor, bool a_rows, bool b_rows,
                             size_t block_m, size_t block_n, size_t block_k, bool edges);

// Whether a plan of the general kernel keeps its tile where it reads the operands a few bytes at
// a time, or goes to the 128 x 128 tile: a larger tile does not fit its registers then, the 64 x 64 tile
// is the faster one until there are 128 x 128 tiles for every compute unit (645 x 584 x 173 x 3, 90 of them, 8.3
// us and 11.2; 1048 x 373 x 723 x 16, 432 of them, 129 and 42; up to 64 rows it reads nothing twice
// and stays).  Skinny problems have been weighed by select_plan.
bool keeps_small_tile(size_t m, size_t n, size_t batch, int block_m, int block_n, size_t cus);

// Estimated-time choice among the compiled variants for a shape without a tuned entry;
// false for shapes it does not cover: extents that are no multiples of 8, unless they stream, and
// K-contiguous rows that do not start on 16 bytes.
// cus: compute units of the GPU the plan is for (0: the GPU the constants were measured on).
bool model_plan(size_t m, size_t n, size_t k, int lc, int la, int lb, launch_plan* out, size_t batch = 1,
                size_t cus = 0);
// The same for the shapes above, and also for other extents (an odd number of tokens, odd
// features), operands copied first where a kernel needs that; false where the nearest tuned entry
// serves as well.
bool model_plan_any_rows(size_t m, size_t n, size_t k, int lc, int la, int lb, launch_plan* out, size_t batch = 1,
                         size_t cus = 0);
// The streaming kernel's plans alone (skinny shapes: one extent at most 128, or small ones:
// at most 2^20 elements of C; K at least 256, a multiple of 8 where an operand is
// K-contiguous), in kernel space (rows x cols, the operands' K-contiguity): the cheapest by
// estimate and its microseconds; false when no compiled variant takes the problem.
bool stream_plan(size_t rows, size_t cols, size_t k, bool a_kmajor, bool b_kmajor, size_t batch, size_t cus,
                 launch_plan* out, double* microseconds);
launch_plan select_plan_from(const tuned_entry* table, size_t count, size_t m, size_t n, size_t k,
                             int type_idx, int lc, int la, int lb);

inline int type_group_of(int type_idx)
{
    return (type_idx == 1 || type_idx == 3) ? 1 : 0;
}

// any_rows: extents whose rows do not start on 16 bytes go to the estimate too.  Its plans for them copy
// operands and cut K where the tables' entries do without; false is for a call that has no memory
// for that.
launch_plan select_plan(size_t m, size_t n, size_t k, int type_idx, int lc, int la, int lb, size_t batch = 1,
                        size_t cus = 0, bool any_rows = true);

} // namespace host
} // namespace rocm_wmma_gemm

#endif
