// Which kernel a product takes (host code only): the one that is expected to finish first, by a model of the time of each.
//
// The constants (microseconds) were fitted to timings of the pinned kernels over 3788 products (1 .. 8192 rows, 128 .. 262144
// columns, K 128 .. 14336, all layouts, round and ragged sizes) and 700 products with the gate/up epilogue, weights from HBM: a
// coordinate search for the least regret, the time of the chosen kernel over that of the fastest one. Over those products
// the choice took 1.6 % longer than the fastest kernel on average (gate/up 0.5 %). perf/gemm_choice.py measures that. Two changes
// since, a third stage of B on the 256x256 tiles and the staggered walk of K under one or two rows of tiles (NT), made kernels 2 - 20 %
// faster without moving the lines between them: over 400 products of one seed 2.0 % before and 2.1 % after, over 3000 of another
// 2.2 % (0.3 % where 256x256 tiles are chosen, NT 17 - 64 rows 1.7 %, 65 - 256 1.2 %, NN and TN up to 16 rows 4.3 %), over 800 drawn
// gate/up products 3.0 %.
//   * A tiled kernel runs in rounds of one workgroup per CU (two for the small tiles) of `K tiles * step + fixed`. The step
//     is set by the CU's intake of 64 bytes per cycle as much as by the matrix instructions (see the tile shapes' rings at
//     MainCfg), and is a sixth (256x128) to twice (32x64) longer where the second operand is too large to stay in the
//     memory-side cache between calls, for tiles up to 128 columns another 5 % where its rows are no whole 128-byte lines.
//   * Ranges of K fill the machine where the tiles of a product do not. Merged by the last workgroup of a tile: a round
//     trip through memory, and one more of 64 KiB per range and 128x128 tile. Merged by a kernel of their own: its launch,
//     and the partial tiles once through memory: the better one for large tiles and more than a few ranges (512 x 4096 x
//     14336 NT, 256x128 tiles in four ranges: 72.0 us against 68.7; 128 x 4096 x 14336, 128x128 in eight: 37.7 / 34.7).
//   * Nothing is faster than its bytes take; how fast each kernel streams a large second operand is a constant of its own. That
//     decides between the small-M kernels and the 64x64 tiles for a few rows against a vocabulary: 8 x 50304 x 4096 NT
//     68.7 us on the former, 80.2 on the latter; 8 x 28672 x 8192 80 / 90; 16 x 28672 x 4096, activation rows in registers,
//     39.7 / 45.5. In layouts NN and TN the small-M kernel takes rounds of 256 workgroups of 64 columns, and the lines of rows
//     that are no whole ones twice: 16 x 28672 x 4096 NN 52 us (64x128 tiles 44), 16 x 50264 x 4096 123 (79); or, up to 16 rows and 16384
//     columns, one round of 128 columns and ranges of K: 16 x 14336 x 4096 24.5 (25.7 without, 64x64 tiles 26), 16 x 4096 x 14336 25.1 (68, split
//     tiles 28.7).
#include <algorithm>
#include <cmath>
#include <cstdint>
#include "mi355_common.h"
#include "mi355_serving_internal.h"

namespace mi355 {

struct ShapeCost {
    int shape, bm, bn, per_cu;
    float step, step_full, fixed;   // K tile alone on its CU, with `per_cu` workgroups there; outside the K loop
    float uncached;                 // factor on the steps for a large second operand
    float rate;                     // bytes per microsecond * 1e-6 at most
};

static KernelChoice cheapest_kernel(int M, int N, int K, bool a_kc, bool b_kc, bool tiles_ok, bool split_ok, bool whole_lines, bool gate_up) {
    static const ShapeCost plain[] = {
        {kTile256x256, 256, 256, 1, 1.028f, 1.028f, 9.30f, 1.442f, 5.14f}, {kTile128x256, 128, 256, 1, .603f, .603f, 5.85f, 1.466f, 5.32f},
        {kTile256x128, 256, 128, 1, .675f, .675f, 7.40f, 1.157f, 5.13f},   {kTile128x128, 128, 128, 1, .429f, .429f, 4.85f, 1.273f, 5.30f},
        {kTileHalf, 64, 128, 1, .316f, .316f, 3.36f, 1.399f, 6.02f},       {kTile64x64, 64, 64, 2, .200f, .409f, 3.11f, 1.387f, 5.27f},
        {kTile32x64, 32, 64, 2, .134f, .306f, 3.45f, 1.909f, 5.28f},       {kDeepRing, 64, 64, 1, .191f, .191f, 3.29f, 1.419f, 5.10f}};
    // with the gate/up epilogue: shapes whose waves hold 64 columns; 64 columns of the interleaved weight are 32 of C
    static const ShapeCost with_gate[] = {
        {kTile256x256, 256, 256, 1, 1.042f, 1.042f, 9.47f, 1.413f, 4.73f}, {kTile128x256, 128, 256, 1, .588f, .588f, 5.83f, 1.435f, 5.77f},
        {kTile256x128, 256, 128, 1, .670f, .670f, 6.34f, 1.207f, 4.71f},   {kTile128x128, 128, 128, 1, .358f, .358f, 5.10f, 1.367f, 5.20f},
        {kTile64x64, 64, 64, 2, .166f, .435f, 2.95f, 1.732f, 6.03f},       {kDeepRing, 64, 64, 1, .194f, .194f, 3.52f, 1.324f, 4.97f}};
    const ShapeCost* const shapes = gate_up ? with_gate : plain;
    const int n_shapes = gate_up ? (int)(sizeof(with_gate) / sizeof(with_gate[0])) : (int)(sizeof(plain) / sizeof(plain[0]));
    static const int ranges[] = {2, 3, 4, 5, 6, 8, 10, 12, 16};
    const bool nt = a_kc && b_kc;
    const float layout = gate_up ? (nt ? .916f : 1.f) : nt ? .884f : a_kc ? 1.f : .910f;
    const float b_bytes = 2.f * (float)N * (float)K, bytes = b_bytes + 2.f * (float)M * ((float)K + (float)N * (gate_up ? .5f : 1.f));
    const bool from_hbm = b_bytes > 20e6f;
    const int ktiles = (K + 63) / 64;
    KernelChoice best;
    best.shape = 0;
    float best_us = 1e30f;
    const auto consider = [&](float us, int shape, int splits, bool own_merge) {
        if (us >= best_us) return;
        best_us = us;
        best.shape = shape;
        best.splits = splits;
        best.own_merge = own_merge;
        best.wide_ranges = 0;
        best.us = us;
    };
    if (M <= 64 && !gate_up) {   // the small-M kernels: workgroups of 16 rows and 64 (layout NT: 16) columns, the whole of K
        const int row_blocks = (M + 15) / 16;
        const float wgs = (float)row_blocks * (float)((N + (nt ? 15 : 63)) / (nt ? 16 : 64)), k = (float)K / 64.f;
        if (nt) {
            const bool rega = N % 16 == 0 && smallm_nt_rega_tpw(M, N / 16, K, 0, 0) > 0;
            const float rate = rega ? 6.12e6f : M <= 8 ? 6.21e6f : 5.94e6f, lines = from_hbm && !whole_lines ? (M <= 8 ? 1.40f : 1.56f) : 1.f;
            const float stream = b_bytes * (1.f + (float)(row_blocks - 1) * 1.02f) * lines / rate;
            consider(fmaxf(2.85f + k * (from_hbm ? 2.53f : 1.f) * .0202f * fmaxf(1.f, wgs * .0057f), fmaxf(stream, wgs * .0053f) + 1.32f), kSmallM, 1, false);
        } else {
            const float stream = b_bytes * (1.f + (float)(row_blocks - 1) * .1f) * (from_hbm && !whole_lines ? 2.04f : 1.f) / 5.7e6f;
            consider(fmaxf(1.67f + ceilf(wgs / 256.f) * (k * (from_hbm ? 1.38f : 1.f) * .169f + .565f), stream + 2.56f), kSmallM, 1, false);
            // 128 columns and as many ranges of K as CUs are left: 1.4 us for a step of 256 rows, 6.1 TB/s, 1.3 times the bytes where rows are no
            // whole lines, 5.4 us beside them; times .92 (TN: .88), as the other kernels' times here come out against those of the same measurement.
            // Of the time without this kernel the choice takes .906 over 165 products of layers' widths (1, 8, 16 rows, 256 .. 16384 columns, K 1024 ..
            // 14336, weights from HBM; at worst 1.067, 1 x 3072 x 2048 NN 7.7 / 8.2) and .969 over 330 drawn ones (at worst 1.18, 16 x 1536 x 10176 NN
            // 12.1 / 14.2, 16 x 1280 x 1536 TN 5.8 / 6.9); .962 where the weight lies in the memory-side cache, which delivers it faster to more
            // workgroups side by side: there 16 x 14336 x 4096 NN takes 21.3 us, 19.4 on 64 columns (from HBM 24.4, 25.6), 16 x 8192 x 2048 TN 8.2, 6.6
            // (from HBM 11.4, 11.4). Where a weight lies is not known here.
            const int n_wide = (N + 127) / 128, ranges_wide = M <= 16 && split_ok ? std::min(8, std::min(256 / n_wide, K / 256)) : 0;
            if (ranges_wide > 1) {
                const float steps = ceilf((float)K / (256.f * (float)ranges_wide));
                const float wide_us = (a_kc ? .92f : .88f) * (5.4f + fmaxf(1.4f * steps, b_bytes * (whole_lines ? 1.f : 1.3f) / 6.1e6f));
                if (wide_us < best_us) {
                    consider(wide_us, kSmallM, 1, false);
                    best.wide_ranges = ranges_wide;
                }
            }
        }
    }
    if (!tiles_ok) return best;
    for (int i = 0; i < n_shapes; ++i) {
        const ShapeCost& c = shapes[i];
        if ((c.shape == kTile32x64 && !a_kc) || (c.shape == kDeepRing && M > 64)) continue;
        // more than half of every tile would be padding (the gate/up epilogue has no 64-row tiles with more than 64 columns)
        if (c.bm > (gate_up ? 128 : 64) && c.bm >= 2 * M) continue;
        const bool half_nt = c.shape == kTileHalf && nt;   // 128x64 for layout NT
        const int bm = half_nt ? c.bn : c.bm, bn = half_nt ? c.bm : c.bn;
        const long tiles = (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
        const bool narrow = c.bm <= 128 && c.bn <= 128;
        const float factor = layout * (from_hbm ? c.uncached * (narrow && !whole_lines && !gate_up ? 1.05f : 1.f) : 1.f);
        const float floor_us = bytes / (c.rate * 1e6f) + (gate_up ? 3.35f : 1.f);
        const auto loop_us = [&](int splits, int per_cu) {
            const float kt = (float)((ktiles + splits - 1) / splits), one = kt * c.step * factor + c.fixed;
            const long wgs = tiles * splits;
            if (per_cu == 1) return (float)((wgs + 255) / 256) * one;
            const float two = kt * c.step_full * factor + c.fixed;
            const long rem = wgs % 512;
            return (float)(wgs / 512) * two + (rem > 256 ? two : rem > 0 ? one : 0.f);
        };
        // (unsplit, the 32x64 tiles run on a ring of eight stages, one workgroup to a CU)
        consider(fmaxf(loop_us(1, c.shape == kTile32x64 ? 1 : c.per_cu), floor_us), c.shape, 1, false);
        if (!split_ok || c.shape == kDeepRing || tiles > 400) continue;
        for (const int s : ranges) {
            if (tiles * s > 1200 || ktiles < 2 * s) break;
            const float us = fmaxf(loop_us(s, c.per_cu), floor_us), tile_kib = (float)(bm * bn) / 256.f;
            const float part_mb = (float)(tiles * s) * tile_kib / 1024.f;
            if (part_mb > 64.f) break;
            if (c.shape != kTile256x256)   // (those have the merge kernel only)
                consider(us + 1.17f + s * tile_kib * (2.f / 64.f) + part_mb * .267f, c.shape, s, false);
            consider(us + 3.91f + part_mb * .418f, c.shape, s, true);
        }
    }
    return best;
}

// The same, remembered for the last few products of the calling thread: going through the candidates takes the host ~0.5 us,
// a tenth of what the smallest products take altogether.
KernelChoice choose_kernel(int M, int N, int K, bool a_kc, bool b_kc, bool tiles_ok, bool split_ok, bool whole_lines, bool gate_up) {
    struct Entry {
        int M = 0, N = 0, K = 0, flags = 0;
        KernelChoice choice;
    };
    static thread_local Entry seen[64];
    const int flags = a_kc | b_kc << 1 | tiles_ok << 2 | split_ok << 3 | gate_up << 4 | whole_lines << 5;
    const uint32_t hash = ((uint32_t)M * 0x9e3779b1u) ^ ((uint32_t)N * 0x85ebca6bu) ^ ((uint32_t)K * 0xc2b2ae35u) ^ (uint32_t)flags * 0x27d4eb2fu;
    Entry& e = seen[hash >> 26];
    if (e.M != M || e.N != N || e.K != K || e.flags != flags) {
        e.choice = cheapest_kernel(M, N, K, a_kc, b_kc, tiles_ok, split_ok, whole_lines, gate_up);
        e.M = M; e.N = N; e.K = K; e.flags = flags;
    }
    return e.choice;
}

// The direct kernel (hgemm_direct.hip) for a product: tiles and ranges of K. A K tile costs a CU .41 us on 64x64 tiles however many of
// them share it (its vector memory path is busy), .99 us on one 128x128 tile and 1.65 on two. An XCD's
// 32 CUs take an eighth of the tiles, of every range, rounded up: 84 tiles in 3 ranges are 252 workgroups, but 33 on most XCDs, and one CU
// of each walks K for two of them (751 x 385 x 8595 NN 42.6 us, copies 32.3; counted over 256 CUs this was expected to take 25).
// Fitted to 2027 timings of 190 products (1 .. 2600 rows, 64 .. 20000 columns, K 40 .. 9000, all layouts, both operands from HBM; rms 6.6 %). The
// choice among these kernels and the aligned copies, copies_pay, takes 1.4 % more than the fastest of them on average, and over 261 other drawn
// products .80 of the time of copies and of the gather that these kernels replaced; slower than those: 269 x 2593 x 3487 NT 29.8 us (26.4),
// 427 x 1393 x 7277 NT 41.3 (37.3), a K just over one tile against many columns (3 x 17073 x 65 NN 7.2, gathered 5.9), K up to 64 by up to 8 %.
KernelChoice choose_direct(int M, int N, int K, int layout, bool split_ok) {
    static const int ranges[] = {1, 2, 3, 4, 6, 8, 12, 16};
    const int ktiles = (K + 63) / 64;
    const float in_mb = 2e-6f * ((float)M + (float)N) * (float)K, out_mb = 2e-6f * (float)M * (float)N, floor_us = (in_mb + out_mb) / 3.48f + 4.34f;
    const float factor = (layout == MI355_GEMM_TN ? .92f : 1.f) * (in_mb > 20.f ? 1.05f : 1.f);
    KernelChoice best;
    best.us = 1e30f;
    for (const int shape : {(int)kDirect64x64, (int)kDirect128x128}) {
        const bool large = shape == kDirect128x128;
        const int bm = large ? 128 : 64;
        if (large && M <= 32) break;
        const long tiles = (long)((M + bm - 1) / bm) * ((N + bm - 1) / bm);
        for (const int s : ranges) {
            const float part_mb = 4e-6f * (float)(tiles * s) * (float)(bm * bm);
            if (s > 1 && (!split_ok || ktiles < 2 * s || part_mb > 48.f)) break;
            const long on_xcd = (tiles + 7) / 8 * s;
            const float per_cu = (float)((on_xcd + 31) / 32);
            const float step = large ? std::fmax(.994f * (float)((on_xcd + 63) / 64), .826f * per_cu) : .41f * per_cu;
            float us = std::fmax((large ? 5.23f : 4.34f) + (float)((ktiles + s - 1) / s) * step * factor, floor_us) + out_mb * (large ? .222f : .522f);
            if (s > 1) us += 1.8f + .38f * part_mb + .11f * (float)s;
            if (us >= best.us) continue;
            best.us = us;
            best.shape = shape;
            best.splits = s;
        }
    }
    return best;
}

}  // namespace mi355
