// Implementation of the shape -> launch plan lookup (plain C++, no device code).
#include "config_select.hpp"

#include <algorithm>

#include <initializer_list>
#include <limits>
#include <vector>

#include "config_generated.hpp"

namespace rocm_wmma_gemm
{
namespace host
{

const tuned_entry* const tuned_table = generated::entries;
const size_t             tuned_count = generated::entry_count;
const model_constants    model_measured
    = {generated::model_compute_units,      generated::model_launch_us,
       generated::model_reduce_us,          generated::model_plane_bytes_per_us,
       generated::model_tile_bytes_per_us,  generated::model_copy_bytes_per_us,
       generated::model_operand_bytes_per_us,
       generated::model_steps,              generated::model_step_count,
       generated::model_stream_constants};

namespace
{
bool same_slot(const tuned_entry& e, int type_group, int la, int lb, int lc)
{
    return e.type_group == type_group && e.layout_a == la && e.layout_b == lb && e.layout_c == lc;
}

// The tuned table by type group and layouts, in the table's order.  A call looks up to six times for
// an entry, each time in one of the 16 slots: with the whole table of 1376 entries walked every time the look-ups
// of a call that ends at the nearest entry took 2 us of host time, which small problems show.
struct tuned_slots
{
    std::vector<tuned_entry> slot[16];
    tuned_slots()
    {
        for(size_t i = 0; i < generated::entry_count; ++i)
        {
            const tuned_entry& e = generated::entries[i];
            slot[index(e.type_group, e.layout_a, e.layout_b, e.layout_c)].push_back(e);
        }
    }
    static int index(int type_group, int la, int lb, int lc)
    {
        return ((type_group & 1) << 3) | ((la & 1) << 2) | ((lb & 1) << 1) | (lc & 1);
    }
};

// The part of a table that a look-up has to see: its slot of the tuned table, all of any other.
void narrow(const tuned_entry*& table, size_t& count, int type_group, int la, int lb, int lc)
{
    if(table == tuned_table && count == tuned_count)
    {
        static const tuned_slots         slots;
        const std::vector<tuned_entry>& s = slots.slot[tuned_slots::index(type_group, la, lb, lc)];
        table                            = s.data();
        count                            = s.size();
    }
}
} // namespace

bool find_exact(const tuned_entry* table, size_t count, size_t m, size_t n, size_t k,
                int type_group, int la, int lb, int lc, launch_plan* out)
{
    narrow(table, count, type_group, la, lb, lc);
    for(size_t i = 0; i < count; ++i)
    {
        const tuned_entry& e = table[i];
        if(e.m == m && e.n == n && e.k == k && same_slot(e, type_group, la, lb, lc))
        {
            *out = e.plan;
            return true;
        }
    }
    return false;
}

bool find_closest(const tuned_entry* table, size_t count, size_t m, size_t n, size_t k,
                  int type_group, int la, int lb, int lc, launch_plan* out)
{
    narrow(table, count, type_group, la, lb, lc);
    bool   any       = false;
    size_t best_kgap = std::numeric_limits<size_t>::max();
    size_t best_k    = 0;
    for(size_t i = 0; i < count; ++i)
    {
        const tuned_entry& e = table[i];
        if(!same_slot(e, type_group, la, lb, lc))
        {
            continue;
        }
        any              = true;
        const size_t gap = e.k > k ? e.k - k : k - e.k;
        if(gap < best_kgap)
        {
            best_kgap = gap;
            best_k    = e.k;
        }
    }
    if(!any)
    {
        return false;
    }
    double best_d = std::numeric_limits<double>::max();
    for(size_t i = 0; i < count; ++i)
    {
        const tuned_entry& e = table[i];
        if(!same_slot(e, type_group, la, lb, lc) || e.k != best_k)
        {
            continue;
        }
        const double dm = static_cast<double>(m) - static_cast<double>(e.m);
        const double dn = static_cast<double>(n) - static_cast<double>(e.n);
        const double d  = dm * dm + dn * dn;
        if(d < best_d)
        {
            best_d = d;
            *out   = e.plan;
        }
    }
    return true;
}

launch_plan heuristic_plan(size_t m, size_t n, size_t k, int lc)
{
    // kernel-space rows/columns (column-major C runs as the transposed problem)
    const size_t rows = lc == 0 ? m : n;
    const size_t cols = lc == 0 ? n : m;
    launch_plan  plan;
    const size_t big_tiles = ((rows + 255) / 256) * ((cols + 255) / 256);
    plan.variant           = (rows >= 256 && cols >= 256 && big_tiles >= 128) ? 1 : 0;
    plan.swizzle           = 4;
    plan.split_k           = 1;
    plan.touch             = 0;
    const size_t bm        = plan.variant == 1 ? 256 : 128;
    const size_t bk        = plan.variant == 1 ? 64 : 32;
    const size_t tiles     = ((rows + bm - 1) / bm) * ((cols + bm - 1) / bm);
    const size_t k_steps   = (k + bk - 1) / bk;
    if(tiles < 128 && k_steps >= 32)
    {
        // too few tiles for 256 CUs: slice K until the chip is covered about twice,
        // keeping at least 8 K steps per slice
        size_t want = (512 + tiles - 1) / tiles;
        size_t cap  = k_steps / 8;
        size_t s    = want < cap ? want : cap;
        if(s > 64)
        {
            s = 64;
        }
        plan.split_k = s < 1 ? 1 : static_cast<int>(s);
    }
    return plan;
}

namespace
{
// Compiled variants as the model sees them.
struct model_variant
{
    int block_m, block_n, block_k, waves_m, waves_n, pipeline;
};
#define RWG_VARIANT(IDX, BM, BN, BK, WM, WN, PIPE) {BM, BN, BK, WM, WN, PIPE},
constexpr model_variant model_variants[] = {
#include "variants.def"
};
#undef RWG_VARIANT

// Microseconds per K tile of 64 with every compute unit at work, and per tile for its
// stores: measured constants (model_measured), one pair per pipeline and tile.
bool step_cost(const model_variant& v, double* step_us, double* item_us)
{
    if(v.block_k != 64)
    {
        return false;
    }
    for(int i = 0; i < model_measured.step_count; ++i)
    {
        const model_step& s = model_measured.steps[i];
        if(s.pipeline == v.pipeline && s.block_m == v.block_m && s.block_n == v.block_n)
        {
            *step_us = s.step_us;
            *item_us = s.item_us;
            return true;
        }
    }
    return false;
}

// Padded copies where a row is not aligned, in microseconds: a launch that the GEMM waits for, and the
// bytes read and written, 5.6 TB/s while they are few, 4.2 over 2.8 GB.  At the 6 us and 3 TB/s
// that regular extents are priced with, copies looked dear and the persistent kernel's large tiles
// cheap: 685 x 4488 x 1944 49 us on 192 x 192, 37 on copies and 128 x 128; 1519 x 2232 x 4536 76 and 58.
double unaligned_copies_us(double bytes)
{
    const double knee = 48.0 * 1024 * 1024;
    return 3.5 + std::min(bytes, knee) / 5.6e6 + std::max(bytes - knee, 0.0) / 3.8e6;
}

// the general kernel's smallest square tile, 64 x 64 x 64
constexpr int small_general_variant = 34;
static_assert(model_variants[small_general_variant].pipeline == 0 && model_variants[small_general_variant].block_m == 64
                  && model_variants[small_general_variant].block_n == 64,
              "small_general_variant names the general kernel's 64 x 64 tile");
static_assert(model_variants[0].pipeline == 0 && model_variants[0].block_m == 128 && model_variants[0].block_n == 128
                  && model_variants[0].block_k == 32,
              "variant 0 is the general kernel's 128 x 128 tile that unaligned operands go to");

size_t ceil_div(size_t a, size_t b)
{
    return (a + b - 1) / b;
}
} // namespace

bool keeps_small_tile(size_t m, size_t n, size_t batch, int block_m, int block_n, size_t cus)
{
    const size_t units  = cus != 0 ? cus : static_cast<size_t>(model_measured.compute_units);
    const bool   skinny = std::min(m, n) <= 128 && std::max(m, n) >= 512;
    return block_m * block_n <= 64 * 64
           && (skinny || std::min(m, n) <= 64 || ceil_div(m, size_t{128}) * ceil_div(n, size_t{128}) * batch < units);
}

operand_copies padded_copies(size_t m, size_t n, size_t k, bool a_kmajor, bool b_kmajor, bool a_rows, bool b_rows,
                             size_t block_m, size_t block_n, size_t block_k, bool edges)
{
    const size_t m_pad = ceil_div(m, edges ? 8 : block_m) * (edges ? 8 : block_m),
                 n_pad = ceil_div(n, edges ? 8 : block_n) * (edges ? 8 : block_n), k_pad = ceil_div(k, block_k) * block_k;
    operand_copies c;
    c.a       = !a_rows || (!edges && !(k_pad == k && m_pad == m));
    c.b       = !b_rows || (!edges && !(k_pad == k && n_pad == n));
    c.lda     = a_kmajor ? (c.a ? k_pad : k) : (c.a ? m_pad : m);
    c.ldb     = b_kmajor ? (c.b ? k_pad : k) : (c.b ? n_pad : n);
    c.elems_a = !c.a ? 0 : c.lda * (!edges ? (a_kmajor ? m_pad : k_pad) : a_kmajor ? m : k);
    c.elems_b = !c.b ? 0 : c.ldb * (!edges ? (b_kmajor ? n_pad : k_pad) : b_kmajor ? n : k);
    const double copied = static_cast<double>(c.elems_a + c.elems_b);
    const double flops  = 2.0 * m * n * k;
    c.pays              = copied > 0.0
             && ((k >= 128 && flops >= copy_pays_flops_aligned * copied)
                 || (flops >= copy_pays_flops * copied
                     && (a_rows && b_rows ? k >= 2048 && std::max(m, n) >= 5120 : k >= 256)));
    return c;
}

// A plan from arithmetic instead of from the nearest tuned shape: for every compiled
// variant of the two pipelines that serve regular shapes, and every way to split, the
// time is estimated as launch + waves of tiles over the CUs x (K tiles x time per K
// tile + stores) + what the split costs in partial sums, and the cheapest wins.  What
// the nearest tuned shape cannot know is how THIS shape's tile count falls on 256 CUs:
// 3584^3 next to the tuned 3072^3 inherited its 192 x 192 tiles (361 of them, two waves
// with the second less than half full) and ran at 0.7 of the 196 tiles of 256 x 256.
// On the 208 tuned entries the model can serve, its pick is on average 2.7 % slower than
// the tuner's, 25 % at worst.
//
// `any_rows`: also for extents that are no multiples of 8 (see model_plan_any_rows).
namespace
{
bool estimated_plan(size_t m, size_t n, size_t k, int lc, int la, int lb, launch_plan* out, size_t batch,
                    size_t cus_of_device, bool any_rows)
{
    const size_t rows = lc == 0 ? m : n;
    const size_t cols = lc == 0 ? n : m;
    // operands in kernel space: a column-major C runs as the transposed problem
    bool a_kmajor = la == 0, b_kmajor = lb == 1;
    if(lc != 0)
    {
        const bool t = a_kmajor;
        a_kmajor     = b_kmajor;
        b_kmajor     = t;
    }
    // K need not be whole K tiles and no extent need be whole tiles: the persistent kernel cuts
    // every ragged edge off itself.  What it needs is operands whose rows start on 16 bytes;
    // one whose rows do not is copied first, where that pays (padded_copies).
    // Skinny against a large operand (decode-like: a few rows against 4096 x 4096 .. 28672
    // x 8192): the plans of the whole-K streaming kernel compete with the others by their
    // estimates, and stand alone for the shapes the others would only take through copies.
    launch_plan stream_best{};
    double      stream_us   = 0.0;
    const bool  have_stream = stream_plan(rows, cols, k, a_kmajor, b_kmajor, batch, cus_of_device, &stream_best, &stream_us);
    const bool   a_rows = (a_kmajor ? k : rows) % 8 == 0, b_rows = (b_kmajor ? k : cols) % 8 == 0;
    const bool   regular = rows % 8 == 0 && cols % 8 == 0 && a_rows && b_rows;
    // (a C that cannot take 16-byte pieces is not the persistent kernel's.  Where that or a copy
    // comes in and 256 x 256 tiles cover half the chip, the nearest tuned entry's large tile serves
    // as well or better: 3000 x 3000 x 3001, all row-major, 79 us against 89; of 247 drawn shapes beyond the line
    // 63 would be more than 5 % slower by the estimate, of 283 below it 7.  Counted for one entry
    // of a batch: what the table would give 64 x 856 x 673 x 1014 is a small tile in 4 slices, 544 us,
    // the estimate 243)
    const bool   pieces  = cols % 8 == 0;
    const size_t device  = cus_of_device != 0 ? cus_of_device : static_cast<size_t>(model_measured.compute_units);
    const bool   few     = ceil_div(rows, size_t{256}) * ceil_div(cols, size_t{256}) < device / 2;
    // (and copies, one more launch, need a K of 256: 441 x 806 x 150 13.4 us with them, 9.9 by the general
    // kernel; 1018 x 222 x 201 13.7 and 12.7; 254 x 773 x 285 14.1 and 15.3; 608 x 177 x 382 14.2 and 17.5)
    const bool   rows_ok = a_rows && b_rows;
    const bool   takes   = regular || (any_rows && (rows_ok ? few || pieces : few && k >= 256));
    if(k < 64 || rows < 16 || cols < 16 || !takes)
    {
        if(have_stream)
        {
            *out = stream_best;
        }
        return have_stream;
    }
    // (the constants are per compute unit at work, so the estimate carries over to a GPU
    // or partition with another count; the tile walk still assumes 8 XCDs)
    const size_t cus                = cus_of_device != 0 ? cus_of_device : static_cast<size_t>(model_measured.compute_units);
    const double launch_us          = model_measured.launch_us;
    const double reduce_us          = model_measured.reduce_us;
    const double plane_bytes_per_us = model_measured.plane_bytes_per_us; // written, then read by reduce_partials
    const double tile_bytes_per_us  = model_measured.tile_bytes_per_us; // split tail, walk by K tile
    // (small planes are paid for in latency, not bandwidth: past 32 MB the rest moves at
    // twice the rate; 8192x1024x8192 cut in two moves 134 MB in ~30 us)
    auto plane_traffic_us = [&](double bytes) {
        const double knee = 32.0 * 1024 * 1024;
        return bytes <= knee ? bytes / plane_bytes_per_us
                             : knee / plane_bytes_per_us + (bytes - knee) / (2.0 * plane_bytes_per_us);
    };
    const double operand_us = static_cast<double>((rows + cols) * k * batch) * 2.0 / model_measured.operand_bytes_per_us;
    const size_t     kt            = ceil_div(k, size_t{64});
    double           best          = 0.0;
    bool             found         = false;
    bool             best_copies_large = false; // the cheapest tiled plan runs on a copy of the larger operand
    const int        count         = static_cast<int>(sizeof(model_variants) / sizeof(model_variants[0]));
    for(int i = 0; i < count; ++i)
    {
        const model_variant& v = model_variants[i];
        double               step = 0.0, item = 0.0;
        if(!step_cost(v, &step, &item))
        {
            continue;
        }
        if(v.pipeline == 5 && !pieces)
        {
            continue;
        }
        const size_t bm = v.block_m, bn = v.block_n;
        if((bm % 128 != 0 && !a_kmajor) || (bn % 128 != 0 && !b_kmajor))
        {
            continue; // not built for this layout
        }
        if((bm >= 192 && rows < 192) || (bn >= 192 && cols < 192))
        {
            continue; // a tile much larger than the problem
        }
        if(v.pipeline == 6 && (bm == 64 || bn == 64) && rows > 128 && cols > 128)
        {
            continue; // the 64-wide tiles are for skinny shapes
        }
        // (batch entries are more tiles: the persistent kernel numbers its items over the
        // whole batch, the others put the batch in grid.y)
        const size_t tm = ceil_div(rows, bm), tn = ceil_div(cols, bn), tiles = tm * tn * batch;
        const double tile_bytes = static_cast<double>(bm * bn) * 4.0;
        // only the persistent kernel takes ragged M, N or K as they are; the others run on
        // padded copies of the operands that need them (one more launch)
        double     copies_us    = 0.0;
        bool       large_copied = false; // the larger operand is
        const bool whole        = v.pipeline == 5 || (tm * bm == rows && tn * bn == cols && kt * 64 == k);
        if(!(rows_ok && whole))
        {
            if(k < 256)
            {
                continue; // (see above)
            }
            const operand_copies copies = padded_copies(rows, cols, k, a_kmajor, b_kmajor, a_rows, b_rows, bm, bn, 64, v.pipeline == 5);
            if(!copies.pays)
            {
                continue; // (the launch takes the general kernel where they do not pay)
            }
            large_copied = cols >= rows ? copies.b : copies.a;
            // (regular extents are priced as in the fit of the constants)
            const double bytes = static_cast<double>(copies.elems_a + copies.elems_b) * static_cast<double>(batch) * 4.0;
            copies_us          = regular ? launch_us + bytes / model_measured.copy_bytes_per_us : unaligned_copies_us(bytes);
        }
        auto consider = [&](double t, int split) {
            t += copies_us;
            if(!found || t < best)
            {
                found        = true;
                best         = t;
                best_copies_large = large_copied;
                out->variant = i;
                out->swizzle = 4;
                out->split_k = split;
                // operands that outgrow the 256 MB memory-side cache and are K-contiguous (both, or
                // one of them with a K of 20480 and more: 8192 x 8192 x 16384 with B row-major loses
                // 2 % to it, x 28672 gains 5 %): the workgroups of the persistent kernel start each
                // group of 8 K tiles at different tiles.  (At 268 MB, 4096 x 4096 x 16384 and
                // 8192^3, the plain walk is level or 3 % ahead; at 335 MB the groups gain 17 %.)
                out->touch = v.pipeline == 5 && (rows + cols) * k * 2 * batch >= (size_t{300} << 20)
                                     && ((a_kmajor && b_kmajor && kt >= 64) || ((a_kmajor || b_kmajor) && kt >= 320))
                                 ? plan_touch_field(0, 0, 8)
                                 : 0;
            }
        };
        // whole tiles
        consider(launch_us + static_cast<double>(ceil_div(tiles, cus)) * (kt * step + item), 1);
        // only the last, partial wave of tiles split
        for(const size_t s : {size_t{2}, size_t{3}, size_t{4}, size_t{6}, size_t{8}})
        {
            if(v.pipeline != 5)
            {
                break;
            }
            if(tiles > cus && tiles % cus != 0 && kt / s >= 4 && (tiles % cus) * s <= cus * 5 / 4)
            {
                // (the slices of the split tiles take one more pass over the CUs, or two
                // when there are more of them than CUs)
                consider(launch_us + static_cast<double>(tiles / cus) * (kt * step + item)
                             + static_cast<double>(ceil_div((tiles % cus) * s, cus)) * (ceil_div(kt, s) * step + item)
                             + reduce_us
                             + (tiles % cus) * s * tile_bytes * 2.0 / tile_bytes_per_us,
                         -static_cast<int>(s));
            }
        }
        // every tile split (few tiles, long K)
        if(tiles < cus)
        {
            for(size_t s = 2; s <= 32; s *= 2)
            {
                if(kt / s < 4)
                {
                    break;
                }
                consider(launch_us + static_cast<double>(ceil_div(tiles * s, cus)) * (ceil_div(kt, s) * step + item)
                             + reduce_us + plane_traffic_us(s * tiles * tile_bytes * 2.0),
                         static_cast<int>(s));
            }
        }
        // the persistent kernel's walk by K tile: for few tiles and a long K only (with
        // many tiles the workgroups of an XCD stop walking K in step and lose each
        // other's operand panels in L2: 7168^3 ran at 950 TFLOP/s this way, 1250 by tile)
        if(v.pipeline == 5 && tiles * 4 <= cus && tiles * kt >= 4 * cus)
        {
            const size_t groups = tiles * kt < cus ? tiles * kt : cus;
            consider(launch_us + ceil_div(tiles * kt, groups) * step + item + reduce_us
                         + groups * 1.25 * tile_bytes * 2.0 / tile_bytes_per_us,
                     -1);
        }
    }
    // The two estimates compete for skinny shapes (up to 128 rows or columns) and for small
    // problems (at most 2^20 elements of C, K up to 4096: 512 x 2048 x 2048 12.2 against 17.8
    // us, 256 x 256 x 1024 8.6 against 12.8), in every layout.  From 65 rows on only while
    // the streaming plan's workgroups all run at once: the estimates are closer to each
    // other than to the truth where they need a second pass over the compute units
    // (128 x 14336 x 4096: 34.5 us streamed, 29.2 tiled; 128 x 8192 x 8192, one pass, 30.3
    // against 37.4), or where the tiled plan would copy the large operand (101 x 22336 x 7808,
    // B row-major: 118 us streamed, 220 on a copy).
    bool one_pass = false;
    if(have_stream)
    {
        const model_variant& v      = model_variants[stream_best.variant];
        const size_t         groups = ceil_div(rows, static_cast<size_t>(v.block_m))
                              * ceil_div(cols, static_cast<size_t>(v.block_n))
                              * static_cast<size_t>(stream_best.split_k) * batch;
        one_pass = groups <= cus * ((v.block_m == 64 && v.block_n == 64) ? 1 : 2);
    }
    const size_t skinny  = std::min(rows, cols);
    const bool   compete = skinny <= 64 || (skinny <= 128 && one_pass)
                         || (rows * cols <= (size_t{1} << 20) && k <= 4096)
                         || (!regular && skinny <= 128 && best_copies_large);
    // Regular, and no tile without copies that are too dear for it: less than 192 rows or columns that are no
    // multiple of 128.  Where the streaming plan does not run in one pass either, or needs a longer K, the
    // general kernel's 64 x 64 tile reads them as they are (128 x 704 x 192 3.4 us, 13.2 on copies and 6.8 on
    // its 128 x 128 tile; 67 x 160 x 200 x 256 8.3 us, 22.3 streamed, 11.4; in one pass 48 x 256 x 512 6.0 and
    // 4.3 streamed).
    if(!found && regular && (!have_stream || (!one_pass && k <= 768)))
    {
        out->variant = small_general_variant;
        out->swizzle = 4;
        out->split_k = 1;
        out->touch   = 0;
        return true;
    }
    // (no tiled plan moves A and B faster than operand_bytes_per_us, which is what bounds the
    // skinny shapes; the estimates above rank the tiled plans among themselves without it)
    const double tiled_us = std::max(best, launch_us + operand_us);
    // (ragged extents with a longer K, where tiles are part empty and some plans copy: from HBM the streaming
    // plan takes 1.6 times its estimate, the tiled ones less than theirs, and the two are level
    // where the estimates are 1 to 2.  391 timed pairs with one workgroup to a streaming tile: 0.86 of
    // the tiled time beyond that ratio, 171 x 1088 x 4800 14 us and 25, 141 x 5440 x 7744 44 and 69; 1.22 below
    // it.  Past a K of 8192 they are level at 1 to 2.5 and only the 64 x 64 tile is worth it, 0.78 of the tiled time
    // beyond (182 x 4288 x 11712 61 us and 84); 32 x 64 gains nothing there, 133 x 5560 x 10232 133 and 89.  Nor do the
    // 16-wide tiles anywhere, 1.15)
    const int  stream_side = !have_stream ? 0 : std::min(model_variants[stream_best.variant].block_m, model_variants[stream_best.variant].block_n);
    const bool stream_late = !regular && skinny > 128 && k > 4096 && have_stream && stream_best.split_k == 1
                             && (k <= 8192 ? stream_side > 16 && 2.0 * stream_us < tiled_us : stream_side >= 64 && 2.5 * stream_us < tiled_us);
    if(have_stream && (!found || stream_late || (stream_us < tiled_us && compete)))
    {
        *out  = stream_best;
        found = true;
    }
    return found;
}
} // namespace

bool model_plan(size_t m, size_t n, size_t k, int lc, int la, int lb, launch_plan* out, size_t batch,
                size_t cus_of_device)
{
    return estimated_plan(m, n, k, lc, la, lb, out, batch, cus_of_device, false);
}

// Any number of tokens against a weight, odd extents: the nearest tuned
// entry knows neither how many tiles there are nor that a small operand is cheap to copy.  Same
// arithmetic, with the copies priced in (133 x 5560 x 10232 134 -> 90 us, 250 x 1001 x 40001 814 -> 75,
// 2001 x 2001 x 16384 321 -> 185; over 1000 drawn shapes 0.73 of the entries' time).
bool model_plan_any_rows(size_t m, size_t n, size_t k, int lc, int la, int lb, launch_plan* out, size_t batch,
                         size_t cus_of_device)
{
    return estimated_plan(m, n, k, lc, la, lb, out, batch, cus_of_device, true);
}

bool stream_plan(size_t rows, size_t cols, size_t k, bool a_kmajor, bool b_kmajor, size_t batch, size_t cus_of_device,
                 launch_plan* out, double* microseconds)
{
    // skinny, or so small that tiles of 64 x 64 do not outnumber the compute units of an MI355X
    // (K in stages of 128, the last of which may be cut short; rows of a K-contiguous operand
    // must stay 16-byte aligned)
    if(k < 256 || ((a_kmajor || b_kmajor) && k % 8 != 0) || rows == 0 || cols == 0
       || (rows > 128 && cols > 128 && rows * cols > (size_t{1} << 20)))
    {
        return false;
    }
    const model_stream& c      = model_measured.stream;
    const size_t        cus    = cus_of_device != 0 ? cus_of_device : static_cast<size_t>(model_measured.compute_units);
    const size_t        stages = (k + 127) / 128;
    const bool          wide   = cols >= rows; // the large operand is B
    const int           count  = static_cast<int>(sizeof(model_variants) / sizeof(model_variants[0]));
    struct stream_candidate
    {
        double us;
        int    variant, slices;
    };
    constexpr int    max_candidates = 32;
    stream_candidate candidate[max_candidates];
    int              candidates = 0;
    for(int i = 0; i < count; ++i)
    {
        const model_variant& v = model_variants[i];
        if(v.pipeline != 7)
        {
            continue;
        }
        const size_t bm = v.block_m, bn = v.block_n;
        if(bm > 64 || bn > 64)
        {
            continue; // the tiles with a 128-wide side are the tuner's to pick: no constants fitted
        }
        // an operand that is not K-contiguous: k rows of 16-byte pieces; on a 32-wide side of
        // the tile (k rows of 64 bytes, half a cache line a request) only while it is skinny
        // and stays in L2 (1024 x 1024 x 4096 with A column-major: 28.4 us on the 32 x 64
        // tile, 18.6 on 64 x 64)
        if((!a_kmajor && (rows % 8 != 0 || (bm <= 32 && rows > 128)))
           || (!b_kmajor && (cols % 8 != 0 || (bn <= 32 && cols > 128))))
        {
            continue;
        }
        const int    slot    = bm == 16 ? (bn == 64 ? 5 : 4) : bn == 16 ? (bm == 64 ? 7 : 6) : (bm == 64 ? 1 : 0) + (bn == 64 ? 2 : 0);
        const size_t tm      = ceil_div(rows, bm), tn = ceil_div(cols, bn), tiles = tm * tn;
        // (transposing reads: by the width of the side they fill, in units of 64)
        const double other   = (a_kmajor ? 0.0 : static_cast<double>(bm) / 64.0) + (b_kmajor ? 0.0 : static_cast<double>(bn) / 64.0);
        const double per_cu  = c.stage_us[slot] * (1.0 + c.transposed_operand * other);
        const double large   = static_cast<double>(wide ? bn : bm) * 256.0;
        const double small   = static_cast<double>(wide ? bm : bn) * 256.0;
        const double sharing = 1.0 + (static_cast<double>(wide ? tm : tn) - 1.0) * c.panel_sharing;
        const bool   large_kmajor = wide ? b_kmajor : a_kmajor, small_kmajor = wide ? a_kmajor : b_kmajor;
        const double rate    = (large_kmajor ? c.bytes_per_us_kmajor : c.bytes_per_us_other)
                            * (!large_kmajor && (wide ? bn : bm) <= 32 ? c.half_line : 1.0)
                            * (std::max(rows, cols) * k * 2 > (size_t{256} << 20) ? (large_kmajor ? c.beyond_cache : c.beyond_cache_other) : 1.0);
        const double l2_rate = c.bytes_per_us_l2 * (!small_kmajor && (wide ? bm : bn) <= 32 ? c.half_line : 1.0);
        for(size_t s = 1; s <= 8; s *= 2)
        {
            // (the counters of the tiles that several workgroups share: 4096 a launch)
            if(stages % s != 0 || stages / s < 2 || (s > 1 && tiles * batch > 4096))
            {
                continue;
            }
            // (the LDS lets two workgroups run on a compute unit at once, one of the 64 x 64 tile)
            const size_t groups   = tiles * s * batch;
            const size_t resident = cus * ((bm == 64 && bn == 64) ? 1 : 2);
            const double active   = static_cast<double>(groups < resident ? groups : resident);
            const double turns  = 1.0 + static_cast<double>(ceil_div(static_cast<size_t>(active), cus) - 1) * c.taking_turns;
            const double stage  = std::max(per_cu * turns, large * (active / sharing) / rate + small * active / l2_rate);
            const double t      = c.launch_us
                             + static_cast<double>(ceil_div(groups, resident)) * (c.fill_us + static_cast<double>(stages / s) * stage)
                             + (s > 1 ? c.exchange_us + c.exchange_us_per_kb * static_cast<double>(s * bm * bn * 4) / 1024.0 : 0.0);
            if(candidates < max_candidates)
            {
                candidate[candidates++] = {t, i, static_cast<int>(s)};
            }
        }
    }
    if(candidates == 0)
    {
        return false;
    }
    // Of the plans whose estimate is within 3 % of the lowest, the one with the fewest
    // workgroups per tile (the exchange is the least certain part of an estimate), then the
    // lowest: 3.0 -> 2.6 % behind the best timed plan on average over the recorded sweep,
    // 32 -> 20 % at worst.
    double lowest = candidate[0].us;
    for(int j = 1; j < candidates; ++j)
    {
        lowest = std::min(lowest, candidate[j].us);
    }
    const stream_candidate* pick = nullptr;
    for(int j = 0; j < candidates; ++j)
    {
        const stream_candidate& x = candidate[j];
        if(x.us <= lowest * 1.03
           && (pick == nullptr || x.slices < pick->slices || (x.slices == pick->slices && x.us < pick->us)))
        {
            pick = &x;
        }
    }
    *microseconds = pick->us;
    out->variant  = pick->variant;
    out->swizzle  = 1;
    out->split_k  = pick->slices;
    out->touch    = 0;
    return true;
}

launch_plan select_plan_from(const tuned_entry* table, size_t count, size_t m, size_t n, size_t k,
                             int type_idx, int lc, int la, int lb)
{
    const int   group = type_group_of(type_idx);
    launch_plan plan;
    if(find_exact(table, count, m, n, k, group, la, lb, lc, &plan))
    {
        return plan;
    }
    if(group != 0 && find_exact(table, count, m, n, k, 0, la, lb, lc, &plan))
    {
        return plan;
    }
    if(find_closest(table, count, m, n, k, group, la, lb, lc, &plan))
    {
        return plan;
    }
    if(group != 0 && find_closest(table, count, m, n, k, 0, la, lb, lc, &plan))
    {
        return plan;
    }
    return heuristic_plan(m, n, k, lc);
}

namespace
{
// What the whole-K streaming kernel asks of a shape (the pointers are the launch's business):
// a stage of K, 16-byte aligned rows of either kind.
bool streaming_takes(size_t m, size_t n, size_t k, int lc, int la, int lb)
{
    const size_t rows = lc == 0 ? m : n, cols = lc == 0 ? n : m;
    bool         a_kmajor = la == 0, b_kmajor = lb == 1;
    if(lc != 0)
    {
        std::swap(a_kmajor, b_kmajor);
    }
    return k >= 128 && ((!a_kmajor && !b_kmajor) || k % 8 == 0) && (a_kmajor || rows % 8 == 0)
           && (b_kmajor || cols % 8 == 0);
}
} // namespace

launch_plan select_plan(size_t m, size_t n, size_t k, int type_idx, int lc, int la, int lb, size_t batch,
                        size_t cus, bool any_rows)
{
    const int   group = type_group_of(type_idx);
    launch_plan plan;
    // the table was tuned on single GEMMs: a batch changes how many tiles there are to
    // spread, which is the model's business
    const auto estimate = any_rows ? &model_plan_any_rows : &model_plan;
    if(batch > 1 && estimate(m, n, k, lc, la, lb, &plan, batch, cus))
    {
        return plan;
    }
    // a tuned entry for exactly this shape first (the reference's order, steps 1 and 2) ...
    if(find_exact(tuned_table, tuned_count, m, n, k, group, la, lb, lc, &plan)
       || (group != 0 && find_exact(tuned_table, tuned_count, m, n, k, 0, la, lb, lc, &plan)))
    {
        return plan;
    }
    // ... fewer than 16 rows (or columns) as 16 of them, where that entry runs on the streaming
    // kernel: the tiles, the workgroups and the bytes moved are the same (rows past M are read
    // as zeros), so the plan tuned for 16 is the plan for 1 to 15
    // (8 x 4096 x 14336: 19.9 us on the entry's 32 x 16 tile, 23.6 on the estimate's pick)
    if(std::min(m, n) < 16 && std::max(m, n) >= 512)
    {
        const size_t m16 = std::max<size_t>(m, 16), n16 = std::max<size_t>(n, 16);
        if((find_exact(tuned_table, tuned_count, m16, n16, k, group, la, lb, lc, &plan)
            || (group != 0 && find_exact(tuned_table, tuned_count, m16, n16, k, 0, la, lb, lc, &plan)))
           && model_variants[plan.variant].pipeline == 7 && streaming_takes(m, n, k, lc, la, lb))
        {
            return plan;
        }
    }
    // ... then the model, and the nearest tuned entry for the rest.  (Not for a batch: the model
    // has declined it above, and one entry priced as if it had the chip to itself would have its K
    // cut for nothing: 128 x 511 x 511 x 4001 in 8 slices, 2048 tiles before any cut.)
    if(batch == 1 && estimate(m, n, k, lc, la, lb, &plan, 1, cus))
    {
        launch_plan nearest;
        const int    pipeline = model_variants[plan.variant].pipeline;
        const size_t elements = m * n;
        const bool   short_sum = pipeline != 7 && std::min(m, n) > 128 && elements > (size_t{1} << 20) && elements <= (size_t{1} << 21) && k <= 2048;
        if(any_rows && (pipeline == 5 || short_sum) && (m % 8 != 0 || n % 8 != 0 || k % 8 != 0)
           && (find_closest(tuned_table, tuned_count, m, n, k, group, la, lb, lc, &nearest)
               || (group != 0 && find_closest(tuned_table, tuned_count, m, n, k, 0, la, lb, lc, &nearest))))
        {
            // A short sum into a million or two elements of C is where the estimate knows least: it prices
            // neither the general kernel nor, beyond a million, the streaming one, which both take
            // ragged extents without copies.  An entry of theirs goes before a tiled plan (1134 x 1032 x 1272,
            // streaming, 18 us and 25 by the estimate, 774 x 2104 x 1104 22 and 26; 1544 x 900 x 608, general, 12
            // and 18, 290 x 4416 x 1792 29 and 37).  Not further: 269 x 4808 x 3816 50 us and 39,
            // 2657 x 1344 x 1088 39 and 24.
            if(short_sum && (model_variants[nearest.variant].pipeline == 7 || model_variants[nearest.variant].pipeline == 0)
               && nearest.split_k <= 1 && streaming_takes(m, n, k, lc, la, lb))
            {
                return nearest;
            }
            // The order of the K tiles within a tile is timed per weight, the estimate only knows
            // groups of 8 from 300 MB on.  A number of rows that no table holds takes the order of
            // the nearest entry where that has one and agrees on the tile and the split: 777 rows
            // against 28672 x 8192 weights, groups of 4, B column-major 372 -> 356 us, row-major (where
            // the estimate has no groups at all) 408 -> 366; 509 rows, in runs, 216 -> 213.  An entry
            // without an order says less: 3001 x 20480 x 10240 is 1007 us in the estimate's groups
            // of 8, 1126 without.
            if(nearest.variant == plan.variant && nearest.split_k == plan.split_k
               && (plan_k_run(nearest.touch) > 0 || plan_k_group(nearest.touch) > 0))
            {
                plan.touch = nearest.touch;
            }
        }
        return plan;
    }
    // A skinny shape that neither has an entry nor suits the model (rows that are not 16-byte
    // aligned): the nearest tuned entry would be a large square's plan, 256 x 256 tiles
    // for a handful of rows.  The general kernel's small tiles, K cut until there are enough
    // workgroups, all of them at once: three of 64 x 64 to a compute unit (8 x 3678 x 3817, odd K: 41.2 us
    // on the 128 x 128 tile with 15 slices, 28.0 on this one with 12), two of 128 x 128.
    // Up to 64 rows the 64 x 64 tile, unless the general kernel has to read element by element throughout:
    // no operand K-contiguous and a K of 1024 (72 shapes, against the entries: 128 x 128 tiles 0.83, 64 x 64
    // 1.04; below, 1242 x 23 x 304 15 us and 12), or a handful of rows against 30 MB and more that are not (8 x 7570 x 2936 30 us and 40, 4 x 2132 x 8269
    // 31 and 35; below, 10 x 1330 x 1786 25 and 15; more rows, 37 x 5133 x 4395 41 and 41, 64 x 6012 x 14831 102
    // and 88; beyond 16384 columns, where two tiles a compute unit are few, 7 x 24345 x 6771 228 and 221).
    // From 65 on it takes two rows of tiles, each of which reads all of
    // the large operand, and the 128 x 128 tile is ahead where it covers the GPU: by its tiles
    // alone (from one to two compute units on: 104 x 986 x 207 x 64 20.8 us, 39.2 on 64 x 64), or cut along a K
    // of 2048 and more (80 x 8192 x 8191, B row-major 76 us against 124; 112 x 16000 x 3003 73 and 67;
    // below that 80 x 8192 x 1001 29 and 25, and 80 x 1500 x 3003, where the slices end at 11, 24 and 19).
    // Where both operands are K-contiguous, which the general kernel reads 16 bytes at a time
    // whatever their alignment, reading the large one twice costs less: only from 64 MB of it on
    // (97 x 13199 x 16899 311 us, 519 on 64 x 64; 85 x 1880 x 5811 32 and 27, 83 x 19047 x 566 32 and 20).
    // A batch brings workgroups of its own.
    if(std::min(m, n) <= 128 && std::max(m, n) >= 512)
    {
        const size_t units = cus != 0 ? cus : static_cast<size_t>(model_measured.compute_units);
        const size_t small = ceil_div(m, size_t{64}) * ceil_div(n, size_t{64}) * batch;
        const size_t large = ceil_div(m, size_t{128}) * ceil_div(n, size_t{128}) * batch;
        const size_t cut   = std::max<size_t>(1, std::min({2 * units / large, k / 256, size_t{64}})); // 8 K steps of 32 a slice
        const size_t skinny = std::min(m, n), weight = std::max(m, n) * k; // (elements of the large operand)
        const bool   a_k = la == 0, b_k = lb == 1; // K-contiguous, whatever the layout of C
        const bool   large_k = n >= m ? b_k : a_k;
        const bool   once   = a_k && b_k && batch == 1 && weight < (size_t{1} << 25);
        const bool   wide   = skinny > 64    ? !once && (large * 2 >= units || (k >= 2048 && large * cut >= units))
                              : batch > 1    ? false
                              : !a_k && !b_k ? k >= 1024
                                             : !large_k && skinny <= 24 && weight >= 15000000 && std::max(m, n) <= 16384;
        plan.variant       = wide ? 0 : small_general_variant;
        plan.swizzle       = 4;
        plan.touch         = 0;
        plan.split_k       = static_cast<int>(wide ? cut : std::max<size_t>(1, std::min({3 * units / small, ceil_div(k, size_t{64}) / 4, size_t{32}})));
        return plan;
    }
    plan = select_plan_from(tuned_table, tuned_count, m, n, k, type_idx, lc, la, lb);
    // (its cut along K was timed on one GEMM: a batch that fills the GPU with whole tiles has no use for it)
    if(batch > 1 && plan.split_k > 1)
    {
        const model_variant& t     = model_variants[plan.variant];
        const size_t         units = cus != 0 ? cus : static_cast<size_t>(model_measured.compute_units);
        if(ceil_div(m, t.block_m) * ceil_div(n, t.block_n) * batch >= units)
        {
            plan.split_k = 1;
        }
    }
    // The nearest entry may be a small problem's, tuned onto the streaming kernel, which
    // wants 16-byte aligned rows of either kind: a
    // shape that does not fit takes the shape heuristic's plan instead.
    const model_variant& v = model_variants[plan.variant];
    if(v.pipeline == 7 && !streaming_takes(m, n, k, lc, la, lb))
    {
        return heuristic_plan(m, n, k, lc);
    }
    return plan;
}

} // namespace host
} // namespace rocm_wmma_gemm
