// fp16 GEMM for gfx950 (MI355X): C[M,N] = op(A) * op(B), fp16 operands, fp32 accumulation in the MFMA
// accumulators, one rounding to fp16 on the store.
//
// Replaces the reference's GEMM ladder (kernels/gemm/pkg/gemm_unified/csrc/{auto,semi,manual}/gemm_*.{cu,cpp});
// the three operand layouts are the ones the reference's op indices use
// (kernels/gemm/test/correct.py:9-15): NN for finegemm_0..11, TN (a stored [K,M]) for 12/16 and NT (b stored
// [N,K]) for 13..15.
//
// Main kernel: one workgroup of 8 waves computes a 256x256 tile of C, K is walked in steps of 64.
//   * global -> LDS staging uses 16-byte direct-to-LDS copies (no VGPR bounce) into a ring of stages (two of A
//     and three of B, 32 KiB each, for the 256x256 tile, three for 128x128, five for 64x128 / 128x64, eight - or four, with two workgroups
//     on a CU - for 64x64); every wave-instruction writes 1 KiB of contiguous LDS, the XOR swizzle is applied on the
//     global-address side.
//     The copies are buffer loads (scalar tile base + one 32-bit lane offset): a global load with 64-bit lane
//     addresses takes about twice as much issue time away from the MFMAs it runs beside, and several times as
//     much when such loads are issued back to back.
//   * a wave issues an instruction every ~5 cycles at best and every ~10 next to its SIMD partner's MFMAs, whatever the
//     instruction, so the K loop is kept short: it is unrolled over the ring, which makes every LDS address a
//     loop-invariant register plus an immediate (A's stages lie one behind the other, then B's, so that one register
//     reaches all stages of an operand) and every copy destination a scalar plus an immediate; the tile bases advance
//     inside their buffer resources; every tile issues the same instructions (the copies of the last tiles run on a
//     resource whose size is set to zero: out of range, nothing is fetched), so the waits never change and the loop has
//     one body per stage. Per K tile and wave of the 256x256 kernel: 64 MFMAs and ~58 other instructions.
//   * where workgroups share nothing but the rows of A, those of different XCDs walk K from different places (kStagger).
//   * K is free: the tile that holds the last K % 64 columns is taken first, by the prologue, whose copies point the lanes at
//     k >= K out of the resource's range (such a copy writes zeros to LDS; where K ends inside a 16-byte chunk, the prologue
//     puts zeros behind it in LDS itself); the loop is the same code for every K.
//   * an operand whose K index is contiguous in memory is read from LDS with ds_read_b128; an operand whose
//     M/N index is contiguous (B in the NN case) is read with the transposing ds_read_b64_tr_b16, so no
//     transpose pass over B is ever made.
//   * each wave owns a 128x64 sub-tile = 8x4 MFMA 16x16x32 blocks (128 fp32 accumulators per lane); with random
//     operands the 16x16x32 instruction sustains a ~14 % higher rate than 32x32x16 under the board's power limit.
//     The MFMA is issued with the B fragment as first operand, i.e. it produces the transposed block, so a
//     lane ends up with 4 consecutive N of one row of C; the epilogue parks the sub-tile in LDS and stores whole
//     128-byte lines.
#include <algorithm>
#include <type_traits>
#include <utility>
#include "hgemm_tiles.h"
#include "mi355_common.h"
#include "mi355_serving_internal.h"
#include "mi355_timeline.h"

namespace mi355 {

// profiling build: per workgroup of hgemm_main_kernel [wall: entry, loop start, loop end, exit; cycles: loop start, loop
// end; K tiles; 0]
MI355_TL(static __device__ unsigned long long hgemm_stamps[timeline::kMaxWorkgroups * timeline::kSlots];
         static hipError_t read_hgemm_stamps(void* dst, size_t bytes) {   // of this translation unit's kernels
             return hipMemcpyFromSymbol(dst, HIP_SYMBOL(hgemm_stamps), bytes < sizeof(hgemm_stamps) ? bytes : sizeof(hgemm_stamps));
         })

// ---------------------------------------------------------------------------------------------------------
// 256x256x64 main kernel
// ---------------------------------------------------------------------------------------------------------

template <bool A_KC, bool B_KC, int BM_, int BN_, int WM_, int WN_, int STAGES = 0>
struct MainCfg {
    static constexpr int BM = BM_, BN = BN_, BK = 64;
    static constexpr int WM = WM_, WN = WN_, NWAVES = WM_ * WN_, NTHREADS = NWAVES * 64;
    static constexpr int TM = BM / WM / 16;  // MFMA 16x16 blocks along M per wave
    static constexpr int TN = BN / WN / 16;  // along N
    // (the description of the layout an operand does not have is never used: it is formed with an extent that exists)
    using ATileK = KContigTile<A_KC ? BM : 256, BK, NWAVES>;
    using ATileM = MNContigTile<A_KC ? 64 : BM, BK, NWAVES>;
    using BTileK = KContigTile<B_KC ? BN : 256, BK, NWAVES>;
    using BTileN = MNContigTile<B_KC ? 64 : BN, BK, NWAVES>;
    static constexpr int A_BYTES = BM * BK * 2;
    static constexpr int B_BYTES = BN * BK * 2;
    static constexpr int STAGE_BYTES = A_BYTES + B_BYTES;
    // 64 KiB stages: two of them fit, and a third one of B (below); the 48 KiB stages of the 128x256 tiles and the 32 KiB stages of the 128x128 tile
    // get a third, which gives every copy one more K tile of time to land (small problems run few tiles per workgroup and are bound by that latency). The narrow tiles
    // serve products with few rows, which are bound by the stream of the weight matrix from HBM: their ring is as deep
    // as 128 KiB of LDS allow (5 stages of 24 KiB, 8 of 16 KiB), so that a CU keeps ~50 KiB of that stream in flight.
    // STAGES > 0 sets the depth (the 64x64 tiles of small products run with four stages, two workgroups to a CU).
    static constexpr int NSTAGE = STAGES > 0 ? STAGES : STAGE_BYTES > 48 * 1024 ? 2 : STAGE_BYTES > 24 * 1024 ? 3 : STAGE_BYTES > 16 * 1024 ? 5 : 8;
    // The 256x256 tiles fill the 160 KiB: 2 x 32 KiB of A, 3 x 32 KiB of B. A copy of B then has two K tiles to land instead of
    // one, and A's, which most workgroups find in L2, wait behind less. Where B (a weight) comes from HBM a K tile takes ~1.1 us to
    // arrive, longer than its matrix instructions (us, 2 stages of both / 3 of B, operands from HBM, in turn on one card): 500 x 28672 x
    // 4096 NT gate/up 110 / 103, 500 x 6144 x 4096 93 / 77, 2048 x 28672 x 4096 gate/up 403 / 376, 8192 x 4096 x 14336 731 / 681, 8192 x 28672
    // x 4096 gate/up 1428 / 1377, 8192^3 NN 798 / 787, NT 807 / 775, TN 803 / 801. The third stage to A instead, on another card, 3 of B / 3
    // of A: 100 / 104, 77 / 88, 8192 x 4096 x 14336 666 / 653, gate/up 1335 / 1335, 8192^3 757 / 749, 751 / 754, 772 / 769: up to 2 % more where
    // the grid is full, 4 - 14 % less under a few rows of tiles; one rule for all sizes takes B. The price: no LDS is left on the CU, so a
    // kernel of another stream that uses any waits for a tile to end (an RMSNorm of 8 rows beside 8192^3 35 us with 128 KiB, 220 now; kernels
    // of over 32 KiB always did, those without LDS do not). (A deeper ring does
    // nothing for the smaller tiles, which already have two or more K tiles in flight: 128x128 tiles with four or five stages, 64x128
    // with six, and 128x256 and 256x128 tiles with a fourth stage of either operand are within 1 % of what they are.)
    static constexpr int NSTAGE_A = NSTAGE, NSTAGE_B = NSTAGE + (STAGE_BYTES > 48 * 1024 ? 1 : 0);
    static constexpr int LDS_BYTES = A_BYTES * NSTAGE_A + B_BYTES * NSTAGE_B;
    static constexpr int A_INSTS = A_BYTES / (NWAVES * 1024);  // 16-byte copies per lane per K tile
    static constexpr int B_INSTS = B_BYTES / (NWAVES * 1024);
    static constexpr int FRAG_SLOTS = TM > TN ? TM : TN;
};

// x < 0 ? -1 : 0 of a wave-uniform value, computed and kept on the scalar unit (written as a shift or a select, the
// compiler may carry the result, and every value formed from it, in vector registers)
__device__ __forceinline__ int sign_mask_scalar(int x) {
    int r;
    asm("s_ashr_i32 %0, %1, 31" : "=s"(r) : "s"(x) : "scc");
    return r;
}

// Map the linear workgroup id to a C tile so that the workgroups resident on one XCD (ids congruent mod 8)
// cover a compact rectangle of tiles: they then share A row-panels and B column-panels in that XCD's L2.
__device__ __forceinline__ void tile_of_block(int bid, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int total = tiles_m * tiles_n;
    constexpr int kXcd = 8;
    // Large grids: the 256 workgroups that run at the same time (ids 256 s .. 256 s + 255, one per CU) take one
    // super-block of 256 tiles, each XCD an 8 x 4 piece of it, and the super-blocks follow one another in serpentine
    // order, so that consecutive ones share their row panels of A or their column panels of B. A super-block reads
    // (16 + 16) or (32 + 8) panels where the same 256 tiles taken as 8 stripes of 8 x 4 from all over the matrix read
    // all 32 row panels: fewer bytes pass through the memory-side cache, and half of them were there a step earlier.
    const int sb_n = tiles_n % 16 == 0 ? 16 : tiles_n % 8 == 0 ? 8 : 0;   // super-block: sb_m x sb_n tiles
    const int sb_m = sb_n ? 256 / sb_n : 0;
    if (sb_n && tiles_m % sb_m == 0 && total >= 512) {
        const int step = bid >> 8, x = bid & 7, j = (bid >> 3) & 31;    // j: this XCD's 32 workgroups of the step
        const int blocks_n = tiles_n / sb_n;
        const int brow = step / blocks_n;
        const int bcol = (brow & 1) ? blocks_n - 1 - step % blocks_n : step % blocks_n;
        const int xcd_cols = sb_n / 4;                                   // XCD pieces side by side in a super-block
        tm = brow * sb_m + (x / xcd_cols) * 8 + (j & 7);
        tn = bcol * sb_n + (x % xcd_cols) * 4 + (j >> 3);
        return;
    }
    // XCD x runs the ids x, x + 8, ..: total / 8 of them, one more if x < total % 8. It gets as many consecutive tiles, also where
    // total is no multiple of 8 (us, ids in order / this: 33 x 50256 x 4096 NN 89.9 / 80.0, 4352^2 x 4096 NN 171 / 163, the
    // 128x256 tiles of 8000 x 8200 x 2048 NT 337 / 256, 1000 x 4160 x 4096 NT 45.7 / 42.7, 33 x 50257 x 4096 NT 91 / 89).
    const int x = bid % kXcd;
    const int t = x * (total / kXcd) + min(x, total % kXcd) + bid / kXcd;
    // grouped ordering: walk down GROUP rows of tiles before moving to the next column
    constexpr int GROUP = 8;
    int group_size = GROUP * tiles_n;
    int g = t / group_size;
    int first_m = g * GROUP;
    int rows = min(GROUP, tiles_m - first_m);
    int in_g = t - g * group_size;
    tm = first_m + in_g % rows;
    tn = in_g / rows;
}

// EPI selects what is stored: 0 = the product; 1 = silu(g) * u for a B operand whose columns alternate between 32 gate
// columns and their 32 up columns (`act_fn(gate_proj(x)) * up_proj(x)`, benchmarks/flashattn-cuda/modeling_llama.py:227,
// with the two projections interleaved in one weight matrix): a wave then holds g and u of the same outputs in its two
// column blocks, at the same accumulator positions, and C has N / 2 columns.
// R (may be null, may be C itself): a residual of C's shape added to the rounded product, `residual + proj(x)` of
// modeling_llama.py:776,781 with the rounding of the unfused sequence (product to T, then the sum to T).
// RAGGED: M and N need not be multiples of the tile, nor of 8, nor K of 8. Copies of rows past the end are redirected to the last row
// (or, for an operand whose M/N index is contiguous, to the last 8 columns of its extent rounded up to a multiple of 8: the
// columns between the extent and that multiple lie in the padding of the operand's rows, because its leading dimension is
// a multiple of 8, and what they hold only reaches rows / columns of the product that are never stored), so every load
// stays inside the matrices' rows; the epilogue stores only what exists: whole 16-byte pieces wherever a row of C starts
// (global memory takes such an access at any element), the last N % 8 columns of a row element by element.
// SPLIT_K: the grid's y index selects one of `splits` ranges of K, whole K tiles each, as equal as that allows, the last one ending
// with K. Without counters a workgroup stores its partial tile as rows of a padded matrix per range and hgemm_merge_kernel adds them.
// With counters it stores its partial tile (fp32, each lane its own accumulators) to `part`, draws a ticket from the tile's counter,
// and the workgroup that draws the last one adds the partial tiles of all ranges, in the order of the ranges (so the sum does
// not depend on which workgroup arrives last), and runs the epilogue. Ordering without a fence, as in the split-KV
// attention kernel: the partial tiles are stored device-coherently (`sc1`), every lane waits for its stores to be
// acknowledged (`s_waitcnt vmcnt(0)`), a workgroup barrier, then one thread draws the ticket with a relaxed device-scope
// atomic (carried out at the memory side); the last workgroup reads the partial tiles with `sc1` loads behind the branch
// on the ticket's value, and sets the counter back to zero for the next launch.
// (the 256x256 tiles are always merged by a kernel of their own: a workgroup alone would read 256 KiB per range, which no choice takes)
template <int BM, int BN>
constexpr bool kOwnMergeOnly = BM * BN == 256 * 256;
template <typename T, bool A_KC, bool B_KC, int BM, int BN, int WM, int WN, int EPI = 0, bool RAGGED = false, int STAGES = 0, int PER_CU = 1,
          bool SPLIT_K = false>
__global__ __launch_bounds__(WM * WN * 64) __attribute__((amdgpu_waves_per_eu(WM * WN / 4, PER_CU * WM * WN / 4)))
void hgemm_main_kernel(const T* __restrict__ A, const T* __restrict__ B,
                                                         T* C, const T* R, int M, int N, int K, long lda,
                                                         long ldb, long ldc, long ldr, float* part, unsigned* counters, int splits) {
    using V8 = typename Elem<T>::v8;
    using V4 = typename Elem<T>::v4;
    using V2 = typename Elem<T>::v2;
    using Cfg = MainCfg<A_KC, B_KC, BM, BN, WM, WN, STAGES>;
    using ATK = typename Cfg::ATileK;
    using ATM = typename Cfg::ATileM;
    using BTK = typename Cfg::BTileK;
    using BTN = typename Cfg::BTileN;
    constexpr int TM = Cfg::TM, TN = Cfg::TN, BK = Cfg::BK;

    MI355_TL(unsigned long long tl_w[4] = {timeline::wall_clock(), 0, 0, 0}; unsigned long long tl_c[2] = {0, 0};)
    extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
    MI355_LDS char* smem = (MI355_LDS char*)smem_raw;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / Cfg::WN;
    const int wn = wave % Cfg::WN;

    int tile_m, tile_n;
    tile_of_block(blockIdx.x, (M + Cfg::BM - 1) / Cfg::BM, (N + Cfg::BN - 1) / Cfg::BN, tile_m, tile_n);
    const long m0 = (long)tile_m * Cfg::BM;
    const long n0 = (long)tile_n * Cfg::BN;
    if constexpr (SPLIT_K) {   // this workgroup's range of K: whole K tiles, the last range ends with K
        const int all = (K + BK - 1) / BK;
        const int t0 = (int)((long)blockIdx.y * all / splits), t1 = (int)((long)(blockIdx.y + 1) * all / splits);
        const long k0 = (long)t0 * BK;
        K = min(K, t1 * BK) - (int)k0;
        A += A_KC ? k0 : k0 * lda;
        B += B_KC ? k0 : k0 * ldb;
    }

    // ---- global -> LDS copy descriptors --------------------------------------------------------------
    // A copy reads (tile base, kept in scalar registers and advanced per K tile) + (this lane's byte offset inside the
    // tile, a loop-invariant 32-bit VGPR) + (copy index * uniform step). Offsets inside a tile fit 32 bits because the
    // launcher only takes leading dimensions below 2^22 elements.
    const char* a_base;
    const char* b_base;
    uint32_t a_lane_off, b_lane_off, a_copy_step, b_copy_step;
    long a_k_step, b_k_step;
    if constexpr (A_KC) {  // A stored [M,K]
        a_base = (const char*)(A + m0 * lda);
        a_lane_off = (uint32_t)(ATK::first_copy_offset(wave, lane, lda) * 2);
        a_copy_step = (uint32_t)(ATK::copy_stride(lda) * 2);
        a_k_step = ATK::ktile_stride(lda) * 2;
    } else {  // A stored [K,M]
        a_base = (const char*)(A + m0);
        a_lane_off = (uint32_t)(ATM::first_copy_offset(wave, lane, lda) * 2);
        a_copy_step = (uint32_t)(ATM::copy_stride(lda) * 2);
        a_k_step = ATM::ktile_stride(lda) * 2;
    }
    if constexpr (B_KC) {  // B stored [N,K]
        b_base = (const char*)(B + n0 * ldb);
        b_lane_off = (uint32_t)(BTK::first_copy_offset(wave, lane, ldb) * 2);
        b_copy_step = (uint32_t)(BTK::copy_stride(ldb) * 2);
        b_k_step = BTK::ktile_stride(ldb) * 2;
    } else {  // B stored [K,N]
        b_base = (const char*)(B + n0);
        b_lane_off = (uint32_t)(BTN::first_copy_offset(wave, lane, ldb) * 2);
        b_copy_step = (uint32_t)(BTN::copy_stride(ldb) * 2);
        b_k_step = BTN::ktile_stride(ldb) * 2;
    }

    // RAGGED: one lane offset per copy, rows / column chunks past the end folded back inside the matrix (never in
    // front of the tile origin: the tile exists, so its first row and its first 8 columns do)
    uint32_t a_voff[RAGGED ? Cfg::A_INSTS : 1];
    uint32_t b_voff[RAGGED ? Cfg::B_INSTS : 1];
    if constexpr (RAGGED) {
        // byte offset from the tile base of copy i of this lane; origin / extent along the tile's M (or N) axis
        auto clamped = [&](long ld, bool k_contig, int rows_per_inst, int chunks_per_row, int rows_per_pass, int i,
                           long origin, long extent, int swz) {
            const int row = wave * rows_per_inst + lane / chunks_per_row + i * rows_per_pass;
            const int chunk = (lane % chunks_per_row) ^ swz;
            if (k_contig) return (uint32_t)(((min(origin + row, extent - 1) - origin) * ld + chunk * 8) * 2);   // row = M/N index
            return (uint32_t)(((long)row * ld + min(origin + chunk * 8, extent - 8) - origin) * 2);              // row = K index
        };
#pragma unroll
        for (int i = 0; i < Cfg::A_INSTS; ++i) {
            if constexpr (A_KC) {
                const int row = wave * ATK::kRowsPerInst + lane / ATK::kChunksPerRow;
                a_voff[i] = clamped(lda, true, ATK::kRowsPerInst, ATK::kChunksPerRow, ATK::kRowsPerPass, i, m0, M, ATK::swz(row));
            } else {
                const int row = wave * ATM::kRowsPerInst + lane / ATM::kChunksPerRow + i * ATM::kRowsPerPass;
                a_voff[i] = clamped(lda, false, ATM::kRowsPerInst, ATM::kChunksPerRow, ATM::kRowsPerPass, i, m0, (M + 7) & ~7, ATM::swz(row));
            }
        }
#pragma unroll
        for (int i = 0; i < Cfg::B_INSTS; ++i) {
            if constexpr (B_KC) {
                const int row = wave * BTK::kRowsPerInst + lane / BTK::kChunksPerRow;
                b_voff[i] = clamped(ldb, true, BTK::kRowsPerInst, BTK::kChunksPerRow, BTK::kRowsPerPass, i, n0, N, BTK::swz(row));
            } else {
                const int row = wave * BTN::kRowsPerInst + lane / BTN::kChunksPerRow + i * BTN::kRowsPerPass;
                b_voff[i] = clamped(ldb, false, BTN::kRowsPerInst, BTN::kChunksPerRow, BTN::kRowsPerPass, i, n0, (N + 7) & ~7, BTN::swz(row));
            }
        }
    }
    // K need not be a multiple of the tile depth: the last K tile, which then holds K % 64 columns (rows) of the
    // operands, is taken FIRST, by the prologue, with copies of its own (below); the loop never sees it.
    const int ktiles = (K + BK - 1) / BK;
    const int k_first = K - (ktiles - 1) * BK;   // depth of that tile: 1 .. 64
    // A weight stored [N,K] under one or two rows of tiles: every workgroup streams 128-byte pieces of its own rows, a row apart,
    // and all of them the same columns at the same time, which keeps part of the memory channels busy and the others waiting.
    // The XCDs therefore start an eighth of K apart from each other and go on at k = 0 behind the last tile. us, in step /
    // this, weights from HBM: 128 x 28672 x 4096 gate/up 53.9 / 48.1, 64 rows 51.7 / 48.2, 32 rows 46.6 / 43.6, 33 x 50257 bf16 87.1 / 82.2, 128 x
    // 18432 45.9 / 43.2, 128 x 8192 x 8192 42.4 / 39.5, 256 x 28672 84.1 / 82.7, 128 x 6144 and 64 x 4096 x 14336 the same; more rows of tiles, and
    // weights stored [K,N], whose rows lie side by side, gain nothing or lose 1-4 %.
    // The order of the 32-bit sums so depends on the XCD a column's tile falls on (a call repeats itself bit for bit): equal weight
    // rows may come out one rounding apart. Against float64 nothing changes (32 products of 17 - 256 rows, fp16 and bf16): relative errors
    // are equal to 5e-7 of themselves, 0.5 % fewer results are other than the exact one rounded.
    constexpr bool kStagger = A_KC && B_KC && !SPLIT_K && BM <= 128 && BN <= 128;
    int before_wrap = ktiles;   // K tiles in front of the one at k = 0 that follows the last
    if (kStagger && M <= 2 * BM && k_first == BK) {
        static_assert(!kStagger || Cfg::NSTAGE_A == Cfg::NSTAGE_B, "whole turns of both rings in front of the wrap");
        const int whole = (ktiles - ktiles * (int)(blockIdx.x & 7) / 8) / Cfg::NSTAGE_A * Cfg::NSTAGE_A;
        if (whole > 0) before_wrap = whole;
    }
    const long first_tile = k_first < BK ? ktiles - 1 : ktiles - before_wrap;   // position along K, in tiles, of the tile taken first
    int4v a_res = make_buffer_resource(a_base + first_tile * a_k_step);
    int4v b_res = make_buffer_resource(b_base + first_tile * b_k_step);

    // ---- LDS fragment read offsets (bytes inside one stage) -------------------------------------------
    // A fragments: TM blocks of 16 rows; B fragments: TN blocks of 16 columns; a K tile is two 32-deep substeps.
    constexpr int NSUB = BK / 32;
    static_assert(NSUB == 2, "the pipeline below is written for two substeps per K tile");
    // LDS layout: the stages of A one behind the other, then those of B. A stage index is a compile-time constant
    // wherever fragments are read (the K loop is unrolled over the ring), so a fragment address is a loop-invariant
    // register plus an immediate offset and the loop holds no address arithmetic. The immediate field of an LDS read
    // reaches 64 KiB: where an operand's ring is longer than that (less the largest offset inside a stage), its stages
    // are grouped into sets within reach, one register per set.
    constexpr int kAImm = A_KC ? (TM - 1) * 16 * ATK::kRowBytes : 36 * ATM::kRowBytes;   // largest offset inside a stage
    constexpr int kBImm = B_KC ? (TN - 1) * 16 * BTK::kRowBytes : 36 * BTN::kRowBytes;
    constexpr int kAPerSet = (65535 - kAImm) / Cfg::A_BYTES + 1, kBPerSet = (65535 - kBImm) / Cfg::B_BYTES + 1;
    constexpr int NSA = Cfg::NSTAGE_A, NSB = Cfg::NSTAGE_B;
    constexpr int kASets = (NSA + kAPerSet - 1) / kAPerSet, kBSets = (NSB + kBPerSet - 1) / kBPerSet;
    constexpr int kBRegion = NSA * Cfg::A_BYTES;
    MI355_LDS char* a_ptr[kASets][Cfg::FRAG_SLOTS];  // K-contiguous operand: one per k-substep; M/N-contiguous: one per 16-wide block
    MI355_LDS char* b_ptr[kBSets][Cfg::FRAG_SLOTS];
#pragma unroll
    for (int s = 0; s < kASets; ++s) {
        MI355_LDS char* base = smem + s * kAPerSet * Cfg::A_BYTES;
        if constexpr (A_KC) {
#pragma unroll
            for (int kk = 0; kk < NSUB; ++kk) a_ptr[s][kk] = base + ATK::frag_offset(wm * TM * 16, kk, lane);
        } else {
#pragma unroll
            for (int i = 0; i < TM; ++i) a_ptr[s][i] = base + ATM::frag_offset(wm * TM * 16 + i * 16, lane);
        }
    }
#pragma unroll
    for (int s = 0; s < kBSets; ++s) {
        MI355_LDS char* base = smem + kBRegion + s * kBPerSet * Cfg::B_BYTES;
        if constexpr (B_KC) {
#pragma unroll
            for (int kk = 0; kk < NSUB; ++kk) b_ptr[s][kk] = base + BTK::frag_offset(wn * TN * 16, kk, lane);
        } else {
#pragma unroll
            for (int j = 0; j < TN; ++j) b_ptr[s][j] = base + BTN::frag_offset(wn * TN * 16 + j * 16, lane);
        }
    }

    float4v acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};

    // Software pipeline, pinned slot by slot (a slot = one MFMA 16x16x32 and what is issued in its shadow;
    // sched_barrier keeps the compiler from moving anything between slots):
    //   * the fragments of the next substep are read during the FIRST slots of the current one, in the order the MFMAs
    //     will need them, so they have landed long before that substep ends and no MFMA waits on a read it has just
    //     issued;
    //   * the barrier that hands over the next K tile sits in front of the last substep: the reads of that substep
    //     were issued a substep earlier, so the wave reaches the barrier with nothing in flight, and goes on with
    //     MFMAs whose operands are already in registers;
    //   * the copies of the tile after next go out during that last substep, spread over its slots, behind the reads of
    //     the next tile's first fragments.
    constexpr int NSLOT = TM * TN;
    constexpr int NFRAG = TM + TN;
    constexpr int NCOPY = Cfg::A_INSTS + Cfg::B_INSTS;
    // fragment f of substep kk, f in the order of first use: A0, B0 .. B(TN-1), A1 .. A(TM-1)
    auto load_frag = [&](auto sc, auto kc, auto fc, V8(&afn)[TM], V8(&bfn)[TN]) {
        constexpr int f = decltype(fc)::value, kk = decltype(kc)::value;
        constexpr int sa = decltype(sc)::value % NSA, sb = decltype(sc)::value % NSB;   // stages of that tile
        constexpr int aset = sa / kAPerSet, ao = (sa % kAPerSet) * Cfg::A_BYTES;   // set, and stage offset inside it
        constexpr int bset = sb / kBPerSet, bo = (sb % kBPerSet) * Cfg::B_BYTES;
        if constexpr (f == 0 || f > TN) {
            constexpr int i = f == 0 ? 0 : f - TN;
            if constexpr (A_KC) {
                afn[i] = Elem<T>::frag(lds_read_b128(a_ptr[aset][kk] + (ao + i * 16 * ATK::kRowBytes)));
            } else {
                half4 lo = lds_read_tr16_b64(a_ptr[aset][i] + (ao + (kk * 32) * ATM::kRowBytes));
                half4 hi = lds_read_tr16_b64(a_ptr[aset][i] + (ao + (kk * 32 + 4) * ATM::kRowBytes));
                afn[i] = Elem<T>::frag(concat(lo, hi));
            }
        } else {
            constexpr int j = f - 1;
            if constexpr (B_KC) {
                bfn[j] = Elem<T>::frag(lds_read_b128(b_ptr[bset][kk] + (bo + j * 16 * BTK::kRowBytes)));
            } else {
                half4 lo = lds_read_tr16_b64(b_ptr[bset][j] + (bo + (kk * 32) * BTN::kRowBytes));
                half4 hi = lds_read_tr16_b64(b_ptr[bset][j] + (bo + (kk * 32 + 4) * BTN::kRowBytes));
                bfn[j] = Elem<T>::frag(concat(lo, hi));
            }
        }
    };
    auto load_frags = [&](auto sc, auto kc, V8(&afn)[TM], V8(&bfn)[TN]) {
        static_for<0, NFRAG>([&](auto fc) { load_frag(sc, kc, fc, afn, bfn); });
    };
    // copy d of a stage lands at (stage, operand, d) + this wave's 1 KiB slice: a scalar register plus an immediate
    const uint32_t wave_lds = (uint32_t)(uintptr_t)(smem + wave * 1024);
    // part selects what is issued: 0 = the whole copy, 1 = only the scalar instruction that points M0 at the destination,
    // 2 = only the load (M0 was set a slot earlier, the matrix instruction in between is the wait state M0 needs)
    auto issue_copy = [&](auto sc, auto dc, auto part) {
        constexpr int d = decltype(dc)::value, pt = decltype(part)::value;
        constexpr bool is_a = d < Cfg::A_INSTS;
        constexpr int st = decltype(sc)::value % (is_a ? NSA : NSB);
        constexpr int e = is_a ? d : d - Cfg::A_INSTS;
        constexpr int dst = is_a ? st * Cfg::A_BYTES + e * Cfg::NWAVES * 1024 : kBRegion + st * Cfg::B_BYTES + e * Cfg::NWAVES * 1024;
        if constexpr (pt == 1) {
            set_m0_at<dst>(wave_lds);
        } else {
            const int4v& res = is_a ? a_res : b_res;
            uint32_t voff, soff = 0u;
            if constexpr (RAGGED && is_a) voff = a_voff[e];
            else if constexpr (RAGGED) voff = b_voff[e];
            else { voff = is_a ? a_lane_off : b_lane_off; soff = e * (is_a ? a_copy_step : b_copy_step); }
            if constexpr (pt == 0) copy16_buffer_to_lds_at<dst>(res, voff, soff, wave_lds);
            else copy16_buffer_to_lds_m0(res, voff, soff);
        }
    };
    // next K tile: the two bases advance inside their resource words (two scalar instructions each; the bases are
    // 48-bit addresses, so the carry into word 1 stays inside its address field)
    auto advance_base = [](int4v& res, long step) {
        const uint64_t b = (((uint64_t)(uint32_t)res[1] << 32) | (uint32_t)res[0]) + (uint64_t)step;
        res[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)b);
        res[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
    };
    // The MFMA is issued with the B fragment as first operand, i.e. it produces the transposed block: lane l ends up
    // with C[m = l % 16][n = 4 (l / 16) .. +3] of the block, 4 consecutive columns of one row.
    // one substep: the MFMAs on (afc, bfc); in slot m, `hook(m)` issues what rides along
    auto substep = [&](const V8(&afc)[TM], const V8(&bfc)[TN], auto&& hook) {
        static_for<0, NSLOT>([&](auto mc) {
            constexpr int m = decltype(mc)::value;
            // boustrophedon order over the wave's blocks: from one MFMA to the next exactly one of the two operand
            // fragments changes (at the end of a row of blocks the B fragment stays and A moves on), which costs less
            // switching energy than changing both; on this power-limited part that is worth 1-1.5 % at 8192^3
            constexpr int i = m / TN, j = (i & 1) ? TN - 1 - m % TN : m % TN;
            acc[i][j] = Elem<T>::mfma16(bfc[j], afc[i], acc[i][j]);
            hook(mc);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    // the fragment reads that ride in slot m: fragments m, m + NSLOT, .. (a wave with a single row or column of blocks has
    // more fragments than MFMAs per substep)
    auto frags_of_slot = [&](auto sc, auto kc, auto mc, V8(&afn)[TM], V8(&bfn)[TN]) {
        constexpr int m = decltype(mc)::value;
        if constexpr (m < NFRAG) load_frag(sc, kc, mc, afn, bfn);
        if constexpr (m + NSLOT < NFRAG) load_frag(sc, kc, std::integral_constant<int, m + NSLOT>{}, afn, bfn);
        static_assert(NFRAG <= 2 * NSLOT, "at most two fragment reads per slot");
    };
    // copy d of a tile goes out in slot d * kCopySpacing of the substep behind the barrier that frees its stage: every
    // second slot where there are that many (buffer loads are cheap to issue in a row, and the earlier a copy leaves the
    // more time it has to land), evenly over the substep otherwise
    constexpr int kCopySpacingNum = NSLOT >= 2 * NCOPY ? 8 : 4 * NSLOT / NCOPY, kCopySpacingDen = 4;
    static_assert((NCOPY - 1) * kCopySpacingNum / kCopySpacingDen < NSLOT, "copies go out within one substep");
    // where a substep has a slot to spare, M0 is set one slot ahead of its load
    constexpr bool kSplitM0 = (NCOPY - 1) * kCopySpacingNum / kCopySpacingDen + 1 < NSLOT;
    auto copies_of_slot = [&](auto sc, auto gc) {   // issue the copies whose slot is g
        constexpr int g = decltype(gc)::value;
        static_for<0, NCOPY>([&](auto dc) {
            constexpr int slot = decltype(dc)::value * kCopySpacingNum / kCopySpacingDen;
            if constexpr (!kSplitM0) {
                if constexpr (slot == g) issue_copy(sc, dc, std::integral_constant<int, 0>{});
            } else {
                if constexpr (slot + 1 == g) issue_copy(sc, dc, std::integral_constant<int, 2>{});
            }
        });
        if constexpr (kSplitM0)
            static_for<0, NCOPY>([&](auto dc) {
                if constexpr (decltype(dc)::value * kCopySpacingNum / kCopySpacingDen == g) issue_copy(sc, dc, std::integral_constant<int, 1>{});
            });
    };
    // Rings of NSA stages of A and NSB of B (NSA, or one more), tile t in stages t % NSA and t % NSB. The prologue fills every stage;
    // in tile kt, behind the barrier, the copies of A's tile kt + NSA, then those of B's tile kt + NSB go into the stages tile kt has
    // just left. At that barrier tile kt+1 must have landed: all but the copies issued behind A's of that tile, those of NSA - 2
    // tiles of A and NSB - 2 of B.
    static_assert(NSB == NSA || NSB == NSA + 1, "the order of the copies, and the wait that counts them");
    constexpr int kUnroll = NSA == NSB ? NSA : NSA * NSB;   // tiles after which both rings are where they were
    V8 af[2][TM], bf[2][TN];
    using Sub0 = std::integral_constant<int, 0>;
    using Sub1 = std::integral_constant<int, 1>;
    // The first tile is the one at the end of K. Its copies fetch nothing for k >= K: such a lane's offset is moved out
    // of the range of the resource (2 GiB for these copies; offsets inside a tile stay below that), and a copy that is
    // out of range writes zeros to LDS. Then the bases go back to k = 0 (with K a multiple of 64 the first tile is the
    // one at k = 0 and the bases move on to the next: the tiles are then walked in memory order).
    {
        constexpr uint32_t kOutOfRange = 0x80000000u;   // with any uniform offset added it stays at or above the range, without wrapping
        a_res[2] = (int)0x80000000u;
        b_res[2] = (int)0x80000000u;
        static_for<0, NCOPY>([&](auto dc) {
            constexpr int d = decltype(dc)::value;
            constexpr bool is_a = d < Cfg::A_INSTS;
            constexpr int e = is_a ? d : d - Cfg::A_INSTS;
            constexpr int dst = is_a ? e * Cfg::NWAVES * 1024 : kBRegion + e * Cfg::NWAVES * 1024;
            uint32_t voff, soff = 0u;
            if constexpr (RAGGED && is_a) voff = a_voff[e];
            else if constexpr (RAGGED) voff = b_voff[e];
            else { voff = is_a ? a_lane_off : b_lane_off; soff = e * (is_a ? a_copy_step : b_copy_step); }
            int k_of_lane;   // first k (inside the tile) of the 16 bytes this lane copies
            if constexpr (is_a ? A_KC : B_KC) {
                using TK = std::conditional_t<is_a, ATK, BTK>;
                const int row = wave * TK::kRowsPerInst + lane / TK::kChunksPerRow;
                k_of_lane = ((lane % TK::kChunksPerRow) ^ TK::swz(row)) * 8;
            } else {
                using TC = std::conditional_t<is_a, ATM, BTN>;
                k_of_lane = wave * TC::kRowsPerInst + lane / TC::kChunksPerRow + e * TC::kRowsPerPass;
            }
            if (k_of_lane >= k_first) voff = kOutOfRange;
            copy16_buffer_to_lds_at<dst>(is_a ? a_res : b_res, voff, soff, wave_lds);
        });
        advance_base(a_res, k_first < BK ? -first_tile * a_k_step : a_k_step);
        advance_base(b_res, k_first < BK ? -first_tile * b_k_step : b_k_step);
    }
    static_for<1, NSB>([&](auto sc) {
        constexpr int t = decltype(sc)::value;
        const int records = sign_mask_scalar(t - ktiles);
        a_res[2] = records;
        b_res[2] = records;
        static_for<0, NCOPY>([&](auto dc) {
            if constexpr (t < NSA || decltype(dc)::value >= Cfg::A_INSTS) issue_copy(sc, dc, std::integral_constant<int, 0>{});
        });
        if constexpr (t < NSA) advance_base(a_res, a_k_step);
        advance_base(b_res, b_k_step);
    });
    wait_vmcnt<Cfg::A_INSTS * (NSA - 1) + Cfg::B_INSTS * (NSB - 1)>();
    __syncthreads();
    if constexpr (RAGGED && (A_KC || B_KC)) {
        if ((k_first & 7) != 0) {   // K ends inside a 16-byte chunk of the rows: zeros for what its copy brought from behind K
            const int chunk = k_first >> 3;
            auto clear = [&](auto tk, MI355_LDS char* stage, int rows) {
                using TK = decltype(tk);
                for (int row = tid; row < rows; row += Cfg::NTHREADS) {
                    MI355_LDS uint16_t* c = (MI355_LDS uint16_t*)(stage + row * TK::kRowBytes + ((chunk ^ TK::swz(row)) << 4));
                    for (int e = k_first & 7; e < 8; ++e) c[e] = 0;
                }
            };
            if constexpr (A_KC) clear(ATK{}, smem, BM);
            if constexpr (B_KC) clear(BTK{}, smem + kBRegion, BN);
            __syncthreads();
        }
    }
    load_frags(Sub0{}, Sub0{}, af[0], bf[0]);

    // One K tile in stage sc (a compile-time constant: the loop below is unrolled over the ring). Every tile issues the
    // same instructions, so the count the waits rely on never changes: once no tile is left to fetch, the copies run on
    // an empty buffer (num_records = 0: out of range, nothing is fetched).
    auto tile = [&](auto sc, int kt) {
        using Next = std::integral_constant<int, (decltype(sc)::value + 1) % kUnroll>;
        substep(af[0], bf[0], [&](auto mc) { frags_of_slot(sc, Sub1{}, mc, af[1], bf[1]); });
        // my copies of the next tile have landed and my reads of this stage are complete; after the barrier that holds
        // for every wave, so this stage may be refilled and the next one may be read
        wait_vmcnt<Cfg::A_INSTS * (NSA - 2) + Cfg::B_INSTS * (NSB - 2)>();
        __syncthreads();
        a_res[2] = sign_mask_scalar(kt + NSA - ktiles);   // -1 while a tile is left to fetch, else 0
        b_res[2] = NSA == NSB ? a_res[2] : sign_mask_scalar(kt + NSB - ktiles);
        substep(af[1], bf[1], [&](auto mc) {
            frags_of_slot(Next{}, Sub0{}, mc, af[0], bf[0]);
            copies_of_slot(sc, mc);   // tiles kt + NSA of A, kt + NSB of B
        });
        advance_base(a_res, a_k_step);
        advance_base(b_res, b_k_step);
    };
    int kt = 0;
    MI355_TL(tl_w[1] = timeline::wall_clock(); tl_c[0] = timeline::shader_cycles();)
    // (the copies run NSA tiles ahead: they go back to k = 0 when the tile NSA in front of the wrap is next)
    for (int stop = before_wrap < ktiles ? before_wrap - NSA : ktiles;; stop = ktiles) {
        for (; kt < stop; kt += kUnroll)
            static_for<0, kUnroll>([&](auto sc) {
                if (kt + decltype(sc)::value < ktiles) tile(sc, kt + decltype(sc)::value);
            });
        if (!kStagger || stop == ktiles) break;
        advance_base(a_res, -ktiles * a_k_step);
        advance_base(b_res, -ktiles * b_k_step);
    }
    MI355_TL(tl_w[2] = timeline::wall_clock(); tl_c[1] = timeline::shader_cycles();)

    // ---- epilogue ------------------------------------------------------------------------------------------------
    constexpr int TNO = EPI == 1 ? TN / 2 : TN;   // column blocks a wave stores
    static_assert(Cfg::NWAVES * TM * 16 * TNO * 32 <= Cfg::LDS_BYTES, "epilogue staging does not fit in LDS");
    wait_vmcnt<0>();  // the last tiles' copies (on the empty buffer) have written their zeros
    __syncthreads();  // every wave has finished reading the operand stages
    if constexpr (SPLIT_K) {
        if (kOwnMergeOnly<BM, BN> || counters == nullptr) {   // the partial tiles are merged by a kernel of their own: [range][padded M][padded N]
            const long np = (long)((N + BN - 1) / BN) * BN, mp = (long)((M + BM - 1) / BM) * BM;
            float* dst = part + ((long)blockIdx.y * mp + m0 + wm * TM * 16 + (lane & 15)) * np + n0 + wn * TN * 16 + 4 * (lane >> 4);
#pragma unroll
            for (int b = 0; b < TM * TN; ++b) *(float4v*)(dst + (long)(b / TN) * 16 * np + (b % TN) * 16) = acc[b / TN][b % TN];
            return;
        }
        // partial tile (tile, range): pair p (two floats) of lane t's accumulator block b at pair (b * 2 + p) * NTHREADS + t,
        // so that every store and load instruction of a wave covers 512 contiguous bytes
        constexpr int NB = TM * TN;
        constexpr long kTilePairs = (long)Cfg::NTHREADS * NB * 2;
        uint64_t* const tile_part = reinterpret_cast<uint64_t*>(part) + (long)blockIdx.x * splits * kTilePairs + tid;
        uint64_t* const mine = tile_part + (long)blockIdx.y * kTilePairs;
        // (device-scope atomic stores, i.e. `global_store_dwordx2 .. sc1`, written as such so that the compiler places the
        // wait states between the last matrix instructions and the first memory instruction that reads their result: a
        // wave that arrives last at the barrier above is only a few cycles behind its last MFMA)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const float4v v = acc[b / TN][b % TN];
                const uint64_t w = (uint64_t)__builtin_bit_cast(uint32_t, (float)v[2 * p]) | (uint64_t)__builtin_bit_cast(uint32_t, (float)v[2 * p + 1]) << 32;
                __hip_atomic_store(mine + (long)(b * 2 + p) * Cfg::NTHREADS, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this lane's part has reached memory before the ticket is drawn
        __syncthreads();
        MI355_LDS unsigned* ticket_sh = (MI355_LDS unsigned*)smem;
        if (tid == 0) *ticket_sh = __hip_atomic_fetch_add(&counters[blockIdx.x], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        const unsigned ticket = *ticket_sh;
        __syncthreads();   // the epilogue below reuses that LDS
        if (ticket != (unsigned)(splits - 1)) return;
        // The last one: every other workgroup of this tile drew its ticket after its part had reached memory. The parts
        // are read with device-coherent loads and added in the order of the ranges, this workgroup's own part too (it is
        // what the registers hold, but a fixed place for it would cost more registers than the load costs time). A batch
        // of loads is a round trip to memory of ~1 us whatever its size, so a batch is as large as the registers allow:
        // 64 registers of a lane, all blocks of one to four ranges.
        constexpr int kChunk = NB < 16 ? NB : 16, kBatch = 16 / kChunk < 4 ? 16 / kChunk : 4;
        static_assert(NB % kChunk == 0, "whole chunks of blocks");
#pragma unroll
        for (int b0 = 0; b0 < NB; b0 += kChunk) {
            float4v sum[kChunk];
#pragma unroll
            for (int b = 0; b < kChunk; ++b) sum[b] = float4v{0.f, 0.f, 0.f, 0.f};
            for (int r0 = 0; r0 < splits; r0 += kBatch) {
                uint64_t v[kBatch][kChunk][2];
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    const uint64_t* pa = tile_part + (long)min(r0 + u, splits - 1) * kTilePairs + (long)b0 * 2 * Cfg::NTHREADS;
#pragma unroll
                    for (int b = 0; b < kChunk * 2; ++b)
                        v[u][b / 2][b % 2] = __hip_atomic_load(pa + (long)b * Cfg::NTHREADS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                __builtin_amdgcn_sched_barrier(0);   // all loads of the batch are issued before the first is waited for
#pragma unroll
                for (int u = 0; u < kBatch; ++u)
                    if (r0 + u < splits)
#pragma unroll
                        for (int b = 0; b < kChunk; ++b)
#pragma unroll
                            for (int q = 0; q < 4; ++q) sum[b][q] += __builtin_bit_cast(float, (uint32_t)(v[u][b][q / 2] >> (32 * (q & 1))));
            }
#pragma unroll
            for (int b = 0; b < kChunk; ++b) acc[(b0 + b) / TN][(b0 + b) % TN] = sum[b];
        }
        if (tid == 0) __hip_atomic_store(&counters[blockIdx.x], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    store_wave_tile<T, TM, TN, EPI, RAGGED>(acc, smem + wave * (TM * 16 * TNO * 32), C, R, m0 + wm * TM * 16,
                                            (EPI == 1 ? n0 / 2 : n0) + wn * TNO * 16, M, EPI == 1 ? N / 2 : N, ldc, ldr, lane);
    MI355_TL(
        wait_vmcnt<0>();   // the stores of this wave have been accepted
        tl_w[3] = timeline::wall_clock();
        if (tid == 0 && blockIdx.x < timeline::kMaxWorkgroups) {
            unsigned long long* rec = hgemm_stamps + (long)blockIdx.x * timeline::kSlots;
            rec[0] = tl_w[0]; rec[1] = tl_w[1]; rec[2] = tl_w[2]; rec[3] = tl_w[3];
            rec[4] = tl_c[0]; rec[5] = tl_c[1]; rec[6] = (unsigned long long)ktiles; rec[7] = 0;
        })
}

// ---------------------------------------------------------------------------------------------------------
// Small-M kernel (decode-shaped GEMM, M <= 16 rows per workgroup row), layouts NN and TN. HBM-bound: B is streamed once.
//   * a workgroup owns 64 columns of C; its 8 waves split K between them (in-workgroup split-K, reduced
//     through LDS at the end, so no global workspace and no atomics);
//   * every wave runs its own copy pipeline, without workgroup barriers: per 32-deep k-step it copies a
//     32x64 slab of B (4 KiB) and a 16x32 slab of A (1 KiB) global -> LDS with 16-byte direct-to-LDS copies,
//     keeps kSmallMStages-1 steps in flight, and waits for the oldest with s_waitcnt vmcnt;
//   * B fragments are read with the transposing LDS read, the product is MFMA 16x16x32;
//   * layout TN (A stored [K,M], A_KC = false): the A slab of a k-step is 32 rows (k) x 16 m, copied as it lies and read
//     with the transposing read like B. Its 16-byte chunks hold 8 rows of the product: the chunks of the rows M .. M
//     rounded up to 8 lie in the padding of A's rows (lda is a multiple of 8 and at least M), their rows of the product
//     are never stored; chunks past that fold back onto the last one.
// ---------------------------------------------------------------------------------------------------------
constexpr int kSmallMWaves = 8;
constexpr int kSmallMStages = 3;
constexpr int kSmallMStageBytes = 5 * 1024;  // 4 KiB of B + 1 KiB of A
constexpr int kSmallMWaveBytes = kSmallMStages * kSmallMStageBytes;
constexpr int kSmallMLdsBytes = kSmallMWaves * kSmallMWaveBytes;
static_assert(kSmallMLdsBytes >= kSmallMWaves * 1024 * 4, "the reduction reuses the pipeline memory");

template <typename T, bool A_KC>
__global__ __launch_bounds__(kSmallMWaves * 64) void hgemm_smallm_nn_kernel(const T* __restrict__ A, const T* __restrict__ B,
                                                              T* C, const T* R, int M, int N, int K, long lda,
                                                              long ldb, long ldc, long ldr, int n_tiles) {
    using V8 = typename Elem<T>::v8;
    using V4 = typename Elem<T>::v4;
    using V2 = typename Elem<T>::v2;
    extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
    MI355_LDS char* smem = (MI355_LDS char*)smem_raw;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // Workgroup i takes column tile i: neighbouring tiles (the 128-byte pieces of one row of B) then run at the same time on
    // different XCDs. Keeping them on one XCD (tile = (i % 8) * (n_tiles / 8) + i / 8) was 3-5 % slower, cached or not
    // (16 x 14336 x 4096: 20.2 -> 19.2 us on a re-read weight, 26.4 -> 25.6 us on one that comes from HBM).
    const int tile = blockIdx.x;
    const int n0 = tile * 64;
    const int m0 = blockIdx.y * 16;

    const int ksteps = K / 32;
    const int s_begin = (int)((long)wave * ksteps / kSmallMWaves);
    const int s_end = (int)((long)(wave + 1) * ksteps / kSmallMWaves);

    MI355_LDS char* wbase = smem + wave * kSmallMWaveBytes;

    // ---- copy descriptors -------------------------------------------------------------------------------
    // B slab: 32 rows (k) x 128 bytes; copy i covers rows 8i .. 8i+7, chunk position lane%8, chunk c of row r
    // is stored at position c ^ 2*(r%4) (keeps the 16 lanes of a transposing read on distinct banks)
    const int b_row = lane >> 3;                                  // + 8*i
    const int b_chunk = (lane & 7) ^ (2 * (b_row & 3));           // (8i + b_row) % 4 == b_row % 4
    const int n_chunk_max = (N + 7) / 8 - 1;   // the last chunk may end in the padding of B's rows
    const int b_col = min(n0 / 8 + b_chunk, n_chunk_max) * 8;     // clamp: columns past N are never stored
    const T* b_src = B + (long)(s_begin * 32 + b_row) * ldb + b_col;
    // A slab: 16 rows (m) x 64 bytes; row lane/4, chunk position lane%4, chunk c of row r at c ^ ((r>>1)&3)
    // A stored [K,M]: slab of 32 rows (k) x 32 bytes; LDS row slot lane/2 holds k row = slot with bits 2 and 3 swapped,
    // which puts the 8 rows that lanes 0..31 of a transposing read touch (k 0..3 and 8..11, + 4 for the second read)
    // into 8 consecutive slots = 256 bytes = distinct banks. Chunks past M fold back onto the last 8 rows of A.
    const int a_row = lane >> 2;
    const int a_chunk = (lane & 3) ^ ((a_row >> 1) & 3);
    const int at_slot = lane >> 1;
    const int at_k = (at_slot & ~12) | ((at_slot & 4) << 1) | ((at_slot & 8) >> 1);
    const T* a_src = A_KC ? A + (long)min(m0 + a_row, M - 1) * lda + (long)s_begin * 32 + a_chunk * 8
                          : A + (long)(s_begin * 32 + at_k) * lda + min(m0 + 8 * (lane & 1), ((M + 7) & ~7) - 8);

    auto issue_stage = [&](int slot) {
        MI355_LDS char* st = wbase + slot * kSmallMStageBytes;
#pragma unroll
        for (int i = 0; i < 4; ++i) copy16_global_to_lds(b_src + (long)(8 * i) * ldb, st + i * 1024);
        copy16_global_to_lds(a_src, st + 4096);
        b_src += 32 * ldb;
        a_src += A_KC ? 32 : 32 * lda;
    };

    // ---- fragment read offsets inside a stage ---------------------------------------------------------------
    // A fragment: lane holds A[m = lane%16][k = 8*(lane/16) .. +7]
    // (A stored [K,M]: transposing read of k rows 8*(lane/16) + 4t + (lane%16)/4, m = 4*(lane%4) .. +3; the second read
    //  (t = 1, k + 4) lies 8 slots = 256 bytes further)
    const int at_read_k = 8 * (lane >> 4) + ((lane & 15) >> 2);
    const int at_read_slot = (at_read_k & ~12) | ((at_read_k & 4) << 1) | ((at_read_k & 8) >> 1);
    const int a_off = A_KC ? 4096 + (lane & 15) * 64 + (((lane >> 4) ^ (((lane & 15) >> 1) & 3)) << 4)
                           : 4096 + at_read_slot * 32 + (lane & 3) * 8;
    // B fragment of column block j: rows 8*(lane/16) + 4t + (lane%16)/4, columns 16j + 4*(lane%4) .. +3
    const int bt_row = 8 * (lane >> 4) + ((lane & 15) >> 2);
    const int bt_swz = 2 * (bt_row & 3);
    int b_off[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        int chunk = (2 * j + ((lane & 3) >> 1)) ^ bt_swz;
        b_off[j] = bt_row * 128 + chunk * 16 + (lane & 1) * 8;
    }

    float4v acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = float4v{0.f, 0.f, 0.f, 0.f};
    auto k_step = [&](MI355_LDS const char* st) {
        V8 af;
        if constexpr (A_KC) af = Elem<T>::frag(lds_read_b128(st + a_off));
        else af = Elem<T>::frag(concat(lds_read_tr16_b64(st + a_off), lds_read_tr16_b64(st + a_off + 256)));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            half4 lo = lds_read_tr16_b64(st + b_off[j]);
            half4 hi = lds_read_tr16_b64(st + b_off[j] + 4 * 128);
            acc[j] = Elem<T>::mfma16(af, Elem<T>::frag(concat(lo, hi)), acc[j]);
        }
    };

    // ---- pipeline ---------------------------------------------------------------------------------------------
    int issued = s_begin;
#pragma unroll
    for (int i = 0; i < kSmallMStages - 1; ++i)
        if (issued < s_end) {
            issue_stage(i);
            ++issued;
        }
    int slot = 0, fill = kSmallMStages - 1;
    for (int s = s_begin; s < s_end; ++s) {
        if (issued < s_end) {
            issue_stage(fill);
            ++issued;
            fill = (fill + 1 == kSmallMStages) ? 0 : fill + 1;
            wait_vmcnt<5 * (kSmallMStages - 1)>();  // everything but the newest kSmallMStages-1 steps has landed
        } else {
            wait_vmcnt<0>();
        }
        k_step(wbase + slot * kSmallMStageBytes);
        slot = (slot + 1 == kSmallMStages) ? 0 : slot + 1;
        // the reads of this slot must be complete before a later copy refills it
        wait_lgkmcnt<0>();
    }
    if (const int k0 = ksteps * 32; k0 < K && wave == kSmallMWaves - 1) {
        // the last K % 32 rows of B (columns of A), by the last wave, whose copies have all landed: zeros behind K
        const int a_left = K - k0 - (A_KC ? 8 * a_chunk : at_k);
        const half8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *(MI355_LDS half8*)(wbase + i * 1024 + lane * 16) = k0 + 8 * i + b_row < K ? *(const half8*)(b_src + (long)(8 * i) * ldb) : zero;
        half8 a_chunk8 = a_left > 0 ? *(const half8*)a_src : zero;
        if (A_KC && (K & 7) != 0) a_chunk8 = first_of_chunk(a_chunk8, a_left);
        *(MI355_LDS half8*)(wbase + 4096 + lane * 16) = a_chunk8;
        wait_lgkmcnt<0>();
        k_step(wbase);
    }

    // ---- reduce the 8 partial tiles through LDS ---------------------------------------------------------------
    // acc[j][q] is D[m = 4*(lane/16) + q][n = 16j + lane%16]
    __syncthreads();  // every wave is done with its staging memory
    MI355_LDS float* red = (MI355_LDS float*)smem;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[wave * 1024 + (4 * (lane >> 4) + q) * 64 + 16 * j + (lane & 15)] = acc[j][q];
    __syncthreads();
    // two columns go out in one 4-byte store where the rows of C (and of the residual) allow it
    const bool pairs = ((reinterpret_cast<uintptr_t>(C) | reinterpret_cast<uintptr_t>(R)) & 3) == 0 && ((ldc | ldr) & 1) == 0;
    for (int o = tid * 2; o < 1024; o += kSmallMWaves * 128) {  // two neighbouring columns of one row
        float s0 = 0.f, s1 = 0.f;
#pragma unroll
        for (int w = 0; w < kSmallMWaves; ++w) {
            s0 += red[w * 1024 + o];
            s1 += red[w * 1024 + o + 1];
        }
        const int m = m0 + (o >> 6);
        const int n = n0 + (o & 63);
        if (m < M && n < N && (n + 1 == N || !pairs)) {
            for (int j = 0; j < 2 && n + j < N; ++j) {
                T v = (T)(j ? s1 : s0);
                if (R != nullptr) v = (T)((float)v + (float)R[(long)m * ldr + n + j]);
                C[(long)m * ldc + n + j] = v;
            }
        } else if (m < M && n < N) {
            V2 v;
            v[0] = (T)s0;
            v[1] = (T)s1;
            if (R != nullptr) {
                const V2 r = *(const V2*)(R + (long)m * ldr + n);
                v[0] = (T)((float)v[0] + (float)r[0]);
                v[1] = (T)((float)v[1] + (float)r[1]);
            }
            *(V2*)(C + (long)m * ldc + n) = v;
        }
    }
}

// The same for a longer K and up to 16384 columns: rows of 256 bytes, which the memory system delivers faster than rows of 128, the
// waves taking k-steps in turn, so that the workgroup reads 256 consecutive rows at a time, and ranges of K (blockIdx.z, at least two) in the
// place of more workgroups side by side. HBM-bound; the ranges are merged by the last workgroup of a tile, in their order (`part` and
// `counters` as in the tiled kernels), which costs ~2 us. us, weights from HBM, what was taken before (this kernel's 64 columns or split
// tiles) / now: 16 x 14336 x 4096 25.5 / 24.5, 16 x 12288 x 4096 25.4 / 22.3, 16 x 6144 x 4096 15.6 / 14.0, 16 x 4096 x 4096 12.4 / 10.9, 16 x 4096 x 14336
// 28.7 / 25.1, 16 x 1024 x 4096 8.9 / 8.1; with K = 1024 the merge costs more than it gives: 16 x 8192 x 1024 7.5 / 8.1.
constexpr int kWideCols = 128;
constexpr int kWideStages = 2;
constexpr int kWideStageBytes = 9 * 1024;   // 8 KiB of B + 1 KiB of A
constexpr int kWideLdsBytes = kSmallMWaves * kWideStages * kWideStageBytes;
constexpr int kWideRed = kWideCols + 4;     // floats between the rows of a wave's partial tile: its four rows of a store lie on different banks
constexpr int kWideRanges = 8;              // at most
static_assert(kWideLdsBytes >= kSmallMWaves * 16 * kWideRed * 4, "the reduction reuses the pipeline memory");
static_assert(kSmallMWaves * 64 * 4 == 16 * kWideCols, "a thread merges and stores four columns of a row");

template <typename T, bool A_KC>
__global__ __launch_bounds__(kSmallMWaves * 64) void hgemm_smallm_wide_kernel(const T* __restrict__ A, const T* __restrict__ B, T* C, const T* R, int M,
                                                                int N, int K, long lda, long ldb, long ldc, long ldr, float* part, unsigned* counters) {
    using V8 = typename Elem<T>::v8;
    using V4 = typename Elem<T>::v4;
    extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
    MI355_LDS char* smem = (MI355_LDS char*)smem_raw;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * kWideCols;
    const int m0 = blockIdx.y * 16;
    const int splits = gridDim.z;
    const int ksteps = K / 32;
    const int r_begin = (int)((long)blockIdx.z * ksteps / splits);
    const int r_end = (int)((long)(blockIdx.z + 1) * ksteps / splits);
    const int first = r_begin + wave, steps = (r_end - first + kSmallMWaves - 1) / kSmallMWaves;   // (no step left: 0, or a quotient rounded up to 0)
    MI355_LDS char* wbase = smem + wave * (kWideStages * kWideStageBytes);

    // B slab: 32 rows (k) x 256 bytes; copy i covers rows 4i .. 4i+3, chunk c of row r at c ^ 2 * (r % 4 + 4 * (r / 8 % 2)): the eight rows
    // and chunk pairs that lanes 0..31 of a transposing read touch lie on distinct banks. A slab as in the kernel above.
    const int b_row = lane >> 4;
    const int n_chunk_max = (N + 7) / 8 - 1;
    const int b_col[2] = {min(n0 / 8 + ((lane & 15) ^ (2 * b_row)), n_chunk_max) * 8, min(n0 / 8 + ((lane & 15) ^ (2 * b_row) ^ 8), n_chunk_max) * 8};
    const int a_row = lane >> 2;
    const int a_chunk = (lane & 3) ^ ((a_row >> 1) & 3);
    const int at_slot = lane >> 1;
    const int at_k = (at_slot & ~12) | ((at_slot & 4) << 1) | ((at_slot & 8) >> 1);
    const auto b_at = [&](int step, int i) { return B + ((long)step * 32 + 4 * i + b_row) * ldb + b_col[(i >> 1) & 1]; };
    const auto a_at = [&](int step) {
        return A_KC ? A + (long)min(m0 + a_row, M - 1) * lda + (long)step * 32 + a_chunk * 8
                    : A + ((long)step * 32 + at_k) * lda + min(m0 + 8 * (lane & 1), ((M + 7) & ~7) - 8);
    };
    const auto issue = [&](int i, int slot) {
        const int step = first + i * kSmallMWaves;
        MI355_LDS char* st = wbase + slot * kWideStageBytes;
#pragma unroll
        for (int c = 0; c < 8; ++c) copy16_global_to_lds(b_at(step, c), st + c * 1024);
        copy16_global_to_lds(a_at(step), st + 8192);
    };

    const int at_read_k = 8 * (lane >> 4) + ((lane & 15) >> 2);
    const int at_read_slot = (at_read_k & ~12) | ((at_read_k & 4) << 1) | ((at_read_k & 8) >> 1);
    const int a_off = A_KC ? 8192 + (lane & 15) * 64 + (((lane >> 4) ^ (((lane & 15) >> 1) & 3)) << 4)
                           : 8192 + at_read_slot * 32 + (lane & 3) * 8;
    const int bt_row = at_read_k;
    const int bt_swz = 2 * ((bt_row & 3) | (((bt_row >> 3) & 1) << 2));
    float4v acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = float4v{0.f, 0.f, 0.f, 0.f};
    const auto k_step = [&](MI355_LDS const char* st) {
        V8 af;
        if constexpr (A_KC) af = Elem<T>::frag(lds_read_b128(st + a_off));
        else af = Elem<T>::frag(concat(lds_read_tr16_b64(st + a_off), lds_read_tr16_b64(st + a_off + 256)));
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            MI355_LDS const char* const p = st + bt_row * 256 + (((2 * j + ((lane & 3) >> 1)) ^ bt_swz) << 4) + (lane & 1) * 8;
            const half4 lo = lds_read_tr16_b64(p), hi = lds_read_tr16_b64(p + 4 * 256);
            acc[j] = Elem<T>::mfma16(af, Elem<T>::frag(concat(lo, hi)), acc[j]);
        }
    };

    // the last K % 32 rows of B (columns of A) go through registers of one wave, zeros behind K: requested in front of its steps, as waiting
    // for them behind the steps costs 2.5 us (2 x 4736 x 3480 13.2)
    const int k0 = ksteps * 32;
    const bool tail = k0 < K && wave == kSmallMWaves - 1 && blockIdx.z == splits - 1;
    half8 tail_b[8] = {}, tail_a = {};
    if (tail) {   // rows behind K: the last one again
#pragma unroll
        for (int c = 0; c < 8; ++c) tail_b[c] = *(const half8*)(B + (long)min(k0 + 4 * c + b_row, K - 1) * ldb + b_col[(c >> 1) & 1]);
        tail_a = *(const half8*)(A_KC ? A + (long)min(m0 + a_row, M - 1) * lda + min(k0 + 8 * a_chunk, (K - 1) & ~7)
                                      : A + (long)min(k0 + at_k, K - 1) * lda + min(m0 + 8 * (lane & 1), ((M + 7) & ~7) - 8));
    }

    static_assert(kWideStages == 2, "one step is in flight while one is worked on");
    if (steps > 0) issue(0, 0);
    for (int i = 0; i < steps; ++i) {
        if (i + 1 < steps) {
            issue(i + 1, (i + 1) & 1);
            wait_vmcnt<9>();
        } else {
            wait_vmcnt<0>();
        }
        k_step(wbase + (i & 1) * kWideStageBytes);
        wait_lgkmcnt<0>();   // the reads of this slot are complete before a later copy refills it
    }
    if (tail) {   // (its steps' copies have all landed)
        const half8 zero = {};
        const int a_left = K - k0 - (A_KC ? 8 * a_chunk : at_k);
        if (A_KC) tail_a = first_of_chunk(tail_a, a_left);
#pragma unroll
        for (int c = 0; c < 8; ++c) *(MI355_LDS half8*)(wbase + c * 1024 + lane * 16) = k0 + 4 * c + b_row < K ? tail_b[c] : zero;
        *(MI355_LDS half8*)(wbase + 8192 + lane * 16) = a_left > 0 ? tail_a : zero;
        wait_lgkmcnt<0>();
        k_step(wbase);
    }

    // the 8 partial tiles through LDS: acc[j][q] is D[m = 4*(lane/16) + q][n = 16j + lane%16]; a thread adds four columns of row tid / 32
    __syncthreads();   // every wave is done with its staging memory
    MI355_LDS float* red = (MI355_LDS float*)smem;
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[(wave * 16 + 4 * (lane >> 4) + q) * kWideRed + 16 * j + (lane & 15)] = acc[j][q];
    __syncthreads();
    float4v sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kSmallMWaves; ++w) sum += *(MI355_LDS const float4v*)(red + (w * 16 + tid / 32) * kWideRed + tid % 32 * 4);
    {
        // partial tile (tile, range): pair p of thread t at pair p * 512 + t; stores, ticket and loads as in hgemm_main_kernel
        constexpr int kPairs = 16 * kWideCols / 2, kThreads = kSmallMWaves * 64;
        const int tile = blockIdx.y * gridDim.x + blockIdx.x;
        uint64_t* const tile_part = reinterpret_cast<uint64_t*>(part) + (long)tile * splits * kPairs + tid;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const uint64_t v = (uint64_t)__builtin_bit_cast(uint32_t, (float)sum[2 * p]) | (uint64_t)__builtin_bit_cast(uint32_t, (float)sum[2 * p + 1]) << 32;
            __hip_atomic_store(tile_part + (long)blockIdx.z * kPairs + p * kThreads, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this lane's part has reached memory before the ticket is drawn
        __syncthreads();
        MI355_LDS unsigned* ticket_sh = (MI355_LDS unsigned*)smem;
        if (tid == 0) *ticket_sh = __hip_atomic_fetch_add(&counters[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*ticket_sh != (unsigned)(splits - 1)) return;
        uint64_t v[kWideRanges][2];   // all ranges in flight together
#pragma unroll
        for (int r = 0; r < kWideRanges; ++r)
#pragma unroll
            for (int p = 0; p < 2; ++p)
                v[r][p] = __hip_atomic_load(tile_part + (long)min(r, splits - 1) * kPairs + p * kThreads, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_sched_barrier(0);
        sum = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < kWideRanges; ++r)
            if (r < splits)
#pragma unroll
                for (int q = 0; q < 4; ++q) sum[q] += __builtin_bit_cast(float, (uint32_t)(v[r][q / 2] >> (32 * (q & 1))));
        if (tid == 0) __hip_atomic_store(&counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const int m = m0 + tid / 32, n = n0 + tid % 32 * 4;
    if (m >= M || n >= N) return;
    T* const c = C + (long)m * ldc + n;
    const T* const r = R + (long)m * ldr + n;
    // four columns go out in one 8-byte store where the rows of C (and of the residual) allow it
    if (n + 4 <= N && ((reinterpret_cast<uintptr_t>(C) | reinterpret_cast<uintptr_t>(R)) & 7) == 0 && ((ldc | ldr) & 3) == 0) {
        V4 v;
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = (T)sum[q];
        if (R != nullptr) {
            const V4 x = *(const V4*)r;
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = (T)((float)v[q] + (float)x[q]);
        }
        *(V4*)c = v;
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (n + q < N) {
                T v = (T)sum[q];
                if (R != nullptr) v = (T)((float)v + (float)r[q]);
                c[q] = v;
            }
    }
}

// hipErrorStreamCaptureUnsupported / hipErrorOutOfMemory: no workspace to be had, the caller takes another kernel.
template <typename T, bool A_KC>
static hipError_t launch_smallm_wide(const T* A, const T* B, T* C, const T* R, int M, int N, int K, long lda, long ldb, long ldc, long ldr, int ranges,
                                     hipStream_t stream) {
    static DynamicLdsOnce lds_once;
    if (hipError_t e = lds_once.ensure(reinterpret_cast<const void*>(hgemm_smallm_wide_kernel<T, A_KC>), kWideLdsBytes); e != hipSuccess) return e;
    ranges = std::min(ranges, kWideRanges);
    const unsigned tiles_n = (N + kWideCols - 1) / kWideCols, tiles_m = (M + 15) / 16;
    const size_t tiles = (size_t)tiles_n * tiles_m;
    if (tiles * sizeof(unsigned) > kSplitKCounterBytes) return hipErrorOutOfMemory;
    char* ws = nullptr;
    std::unique_lock<std::mutex> order;
    if (hipError_t e = split_k_workspace(kSplitKCounterBytes + tiles * ranges * (16 * kWideCols * 4), stream, &ws, &order); e != hipSuccess) return e;
    hgemm_smallm_wide_kernel<T, A_KC><<<dim3(tiles_n, tiles_m, ranges), dim3(kSmallMWaves * 64), kWideLdsBytes, stream>>>(
        A, B, C, R, M, N, K, lda, ldb, ldc, ldr, reinterpret_cast<float*>(ws + kSplitKCounterBytes), reinterpret_cast<unsigned*>(ws));
    return hipGetLastError();
}

template <typename T, bool A_KC>
static hipError_t launch_smallm_nn(const T* A, const T* B, T* C, const T* R, int M, int N, int K, long lda, long ldb,
                                   long ldc, long ldr, hipStream_t stream) {
    static DynamicLdsOnce lds_once;
    if (hipError_t e = lds_once.ensure(reinterpret_cast<const void*>(hgemm_smallm_nn_kernel<T, A_KC>), kSmallMLdsBytes); e != hipSuccess) return e;
    const int n_tiles = (N + 63) / 64;
    dim3 grid(n_tiles, (M + 15) / 16);
    hgemm_smallm_nn_kernel<T, A_KC><<<grid, dim3(kSmallMWaves * 64), kSmallMLdsBytes, stream>>>(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, n_tiles);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------------
// Small-M kernel for layout NT (B stored [N,K]: the nn.Linear weight layout of decode-time projections), M <= 16
// rows per workgroup row. HBM-bound like hgemm_smallm_nn_kernel and built the same way: a workgroup owns 16
// columns of C (16 rows of B), its waves split K and are reduced through LDS; every wave runs a private,
// barrier-free copy pipeline of 64-deep k-steps (16x64 of B and 16x64 of A, 2 KiB each, direct-to-LDS), both
// operands are K-contiguous so both fragments are plain ds_read_b128, the product is MFMA 16x16x32.
// Four waves with four stages each = 64 KiB of LDS, so that two or three workgroups share a CU and one's start-up
// and reduction hide under the others' streaming: with weights that come from HBM (not from the memory-side cache, as
// when one weight matrix is launched on again and again) that beats eight waves on 128 KiB, one workgroup per CU, by
// 7-15 % (8 x 4096 x 14336: 21.7 us against 23.3, 8 x 6144 x 4096: 11.9 against 13.4).
// ---------------------------------------------------------------------------------------------------------
constexpr int kSmallMNtWaves = 4;
constexpr int kSmallMNtStages = 4;
constexpr int kSmallMNtStageBytes = 4 * 1024;  // 2 KiB of B + 2 KiB of A
constexpr int kSmallMNtWaveBytes = kSmallMNtStages * kSmallMNtStageBytes;
constexpr int kSmallMNtLdsBytes = kSmallMNtWaves * kSmallMNtWaveBytes;
static_assert(kSmallMNtLdsBytes >= kSmallMNtWaves * 256 * 4, "the reduction reuses the pipeline memory");

// GATE_UP: the rows of B come in groups of [32 gate | 32 up] (the operand of the tiled kernels' gate/up epilogue) and C is
// silu(gate) * up, half as wide. Workgroup t then takes the 8 gate rows 64 (t / 4) + 8 (t % 4) .. +7 and the 8 up rows 32
// further on, and stores the 8 columns 32 (t / 4) + 8 (t % 4) .. +7 of C.
// kEpiRope: the rows of B are the heads of a fused QKV projection, 128 each. Workgroup t takes 8 rows of the lower half of head
// t / 8 and their partners 64 rows further on, rounds the sums as the plain product stores them, rotates the pairs and writes
// query heads into C, key and value heads where rope.kv_out says: what rope_kernel (glue.hip) makes of the stored product, bit for
// bit, without its launch and its round trip through memory.
enum SmallMEpilogue { kEpiPlain, kEpiGateUp, kEpiRope };
struct NoEpilogueArgs {};
template <int EPI>
using EpilogueArgs = std::conditional_t<EPI == kEpiRope, RopeEpilogue, NoEpilogueArgs>;

// first of the 16 weight rows of tile t, and how far its second 8 rows lie behind its first 8
template <int EPI>
__device__ __forceinline__ int smallm_nt_first_row(int t) {
    return EPI == kEpiGateUp ? 64 * (t >> 2) + 8 * (t & 3) : EPI == kEpiRope ? 128 * (t >> 3) + 8 * (t & 7) : t * 16;
}
template <int EPI>
constexpr int kSmallMNtSecondRows = EPI == kEpiGateUp ? 32 : EPI == kEpiRope ? 64 : 8;

// Column pair e % 16 (< 8) and 8 further on of tile t, row m: `lo` and `hi` are the finished sums.
template <typename T>
__device__ __forceinline__ void store_rope_pair(const RopeEpilogue& rope, T* C, long ldc, int t, int m, int col, float lo_sum, float hi_sum) {
    const int head = t >> 3, i = 8 * (t & 7) + col;
    const int b = m / rope.S, tok = m - b * rope.S;
    T* dst = head < rope.q_heads ? C + (long)m * ldc + (long)head * 128 + i
                                 : static_cast<T*>(rope.kv_out) + b * rope.o_batch + tok * rope.o_row + (head - rope.q_heads) * rope.o_head + i;
    T lo = (T)lo_sum, hi = (T)hi_sum;
    if (head < rope.q_heads + rope.kv_heads) {
        const int pos = min(max(rope.positions[b * rope.pos_batch + tok], 0), rope.n_pos - 1);
        const float c = rope.cos_t[(long)pos * 64 + i], sn = rope.sin_t[(long)pos * 64 + i];
        const float x = (float)lo, y = (float)hi;
        lo = (T)(x * c - y * sn);
        hi = (T)(y * c + x * sn);
    }
    dst[0] = lo;
    dst[64] = hi;
}

// NORM = 1, 2, 4 or 8 (M <= NORM, K >= 1024 and a multiple of 512): A is the residual stream, and what is multiplied is its RMSNorm,
// norm_weight * a * rsqrt(mean(a^2) + eps), rounded as rmsnorm_kernel (glue.hip) rounds it and with its order of summation. A
// workgroup copies the rows and the norm weight into LDS in front of its first weights, normalises them there while those are
// on their way, and reads its A fragments from there: the ring holds weights only. (The number of rows is a constant so that the rows'
// reductions run side by side; rows behind M repeat the last one.)
template <int NORM>
constexpr int kSmallMNtStage = NORM > 0 ? 2 * 1024 : kSmallMNtStageBytes;
constexpr int kNormRowPad = 64;   // bytes behind a row in LDS: the 64 bytes that four rows read together lie in different banks
constexpr int kNormLdsMax = 80 * 1024;   // two workgroups to a CU
static int smallm_nt_norm_rows(int M) { return M <= 2 ? M : M <= 4 ? 4 : 8; }
static int smallm_nt_norm_lds(int M, int K) { return kSmallMNtWaves * kSmallMNtStages * kSmallMNtStage<1> + (smallm_nt_norm_rows(M) + 1) * (2 * K + kNormRowPad); }

template <typename T, bool HALF_A, int EPI, int NORM = 0>
__global__ __launch_bounds__(kSmallMNtWaves * 64) void hgemm_smallm_nt_kernel(const T* __restrict__ A, const T* __restrict__ B,
                                                              T* C, const T* R, int M, int N, int K, long lda,
                                                              long ldb, long ldc, long ldr, int n_tiles, EpilogueArgs<EPI> epi,
                                                              const T* __restrict__ norm_weight, float eps) {
    constexpr bool GATE_UP = EPI == kEpiGateUp;
    constexpr int kStageBytes = kSmallMNtStage<NORM>;
    using V8 = typename Elem<T>::v8;
    using V4 = typename Elem<T>::v4;
    using V2 = typename Elem<T>::v2;
    extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
    MI355_LDS char* smem = (MI355_LDS char*)smem_raw;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    int tile = blockIdx.x;
    if (n_tiles % 8 == 0) tile = (blockIdx.x % 8) * (n_tiles / 8) + blockIdx.x / 8;
    const int n0 = tile * 16;
    const int m0 = blockIdx.y * 16;

    const int ksteps = K / 64;
    const int s_begin = (int)((long)wave * ksteps / kSmallMNtWaves);
    const int s_end = (int)((long)(wave + 1) * ksteps / kSmallMNtWaves);
    MI355_LDS char* wbase = smem + wave * kSmallMNtStages * kStageBytes;

    // slab = 16 rows x 128 bytes; a copy instruction covers 8 rows (row lane/8, chunk position lane%8);
    // chunk c of row r is stored at position c ^ (r & 7)
    const int c_row = lane >> 3;  // + 8*i
    const int c_chunk = (lane & 7) ^ (c_row & 7);
    const int b_row0 = smallm_nt_first_row<EPI>(tile) + c_row;
    const int b_row1 = b_row0 + kSmallMNtSecondRows<EPI>;
    const T* b_src0 = B + (long)min(b_row0, N - 1) * ldb + (long)s_begin * 64 + c_chunk * 8;
    const T* b_src1 = B + (long)min(b_row1, N - 1) * ldb + (long)s_begin * 64 + c_chunk * 8;
    const T* a_src0 = A + (long)min(m0 + c_row, M - 1) * lda + (long)s_begin * 64 + c_chunk * 8;
    const T* a_src1 = A + (long)min(m0 + c_row + 8, M - 1) * lda + (long)s_begin * 64 + c_chunk * 8;

    // HALF_A (M <= 8): rows 8..15 of the A slab are not copied; the fragment rows read from there hold whatever the
    // memory held, and so do rows 8..15 of the product, which are never stored (an output row depends on its own A row only)
    constexpr int kCopies = NORM > 0 ? 2 : HALF_A ? 3 : 4;
    auto issue_stage = [&](int slot) {
        MI355_LDS char* st = wbase + slot * kStageBytes;
        copy16_global_to_lds(b_src0, st);
        copy16_global_to_lds(b_src1, st + 1024);
        if constexpr (NORM == 0) copy16_global_to_lds(a_src0, st + 2048);
        if constexpr (NORM == 0 && !HALF_A) copy16_global_to_lds(a_src1, st + 3072);
        b_src0 += 64;
        b_src1 += 64;
        a_src0 += 64;
        a_src1 += 64;
    };

    // fragment of k-substep sub (32 deep): lane holds X[row = lane%16][k = 32*sub + 8*(lane/16) .. +7]
    const int f_row = lane & 15;
    int f_off[2];
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) f_off[sub] = f_row * 128 + (((4 * sub + (lane >> 4)) ^ (f_row & 7)) << 4);

    // NORM: the normalised rows lie behind the ring, one behind the other, then the norm weight
    MI355_LDS char* const rows = smem + kSmallMNtWaves * kSmallMNtStages * kStageBytes;
    const int row_bytes = 2 * K + kNormRowPad;
    MI355_LDS const char* a_norm = rows + min(f_row, NORM - 1) * row_bytes + s_begin * 128 + ((lane >> 4) << 4);

    float4v acc = float4v{0.f, 0.f, 0.f, 0.f};
    auto k_step = [&](MI355_LDS const char* st) {
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            V8 bf = Elem<T>::frag(lds_read_b128(st + f_off[sub]));
            V8 af = Elem<T>::frag(lds_read_b128(NORM > 0 ? a_norm + 64 * sub : st + 2048 + f_off[sub]));
            acc = Elem<T>::mfma16(af, bf, acc);
        }
        if constexpr (NORM > 0) a_norm += 128;
    };

    // in pieces of 512 values, piece p of each by wave p % 4
    const int pieces = K / 512;
    if constexpr (NORM > 0) {
        for (int p = wave; p < pieces; p += kSmallMNtWaves)
#pragma unroll
            for (int r = 0; r <= NORM; ++r)
                copy16_global_to_lds((r < NORM ? A + (long)min(r, M - 1) * lda : norm_weight) + lane * 8 + p * 512, rows + r * row_bytes + p * 1024);
    }
    int issued = s_begin;
#pragma unroll
    for (int i = 0; i < kSmallMNtStages - 1; ++i)
        if (issued < s_end) {
            issue_stage(i);
            ++issued;
        }
    if constexpr (NORM > 0) {
        // a wave has at least four steps (K >= 1024), so exactly the copies of three stages were issued behind its own pieces
        wait_vmcnt<kCopies * (kSmallMNtStages - 1)>();
        asm volatile("" ::: "memory");
        MI355_LDS char* const mine = rows + wave * 1024 + lane * 16;
        float ss[NORM];
#pragma unroll
        for (int r = 0; r < NORM; ++r) ss[r] = 0.f;
        for (int p = 0; p * kSmallMNtWaves + wave < pieces; ++p) {
            V8 v[NORM];
#pragma unroll
            for (int r = 0; r < NORM; ++r) v[r] = Elem<T>::frag(lds_read_b128(mine + r * row_bytes + p * (kSmallMNtWaves * 1024)));
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int r = 0; r < NORM; ++r) ss[r] += (float)v[r][j] * (float)v[r][j];
        }
        __shared__ float scratch[NORM][kSmallMNtWaves];
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1)
#pragma unroll
            for (int r = 0; r < NORM; ++r) ss[r] += __shfl_xor(ss[r], off, 64);
        if (lane == 0)
#pragma unroll
            for (int r = 0; r < NORM; ++r) scratch[r][wave] = ss[r];
        // (the barriers are written out: __syncthreads() may wait for the weights in flight)
        asm volatile("" ::: "memory");
        wait_lgkmcnt<0>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int r = 0; r < NORM; ++r) {
            const float total = scratch[r][0] + scratch[r][1] + scratch[r][2] + scratch[r][3];
            ss[r] = __builtin_amdgcn_rsqf(total / (float)K + eps);
        }
        for (int p = 0; p * kSmallMNtWaves + wave < pieces; ++p) {
            V8 v[NORM + 1];
#pragma unroll
            for (int r = 0; r <= NORM; ++r) v[r] = Elem<T>::frag(lds_read_b128(mine + r * row_bytes + p * (kSmallMNtWaves * 1024)));
#pragma unroll
            for (int r = 0; r < NORM; ++r) {
                V8 o;
#pragma unroll
                for (int j = 0; j < 8; ++j) o[j] = (T)((float)v[NORM][j] * ((float)v[r][j] * ss[r]));
                *(MI355_LDS V8*)(mine + r * row_bytes + p * (kSmallMNtWaves * 1024)) = o;
            }
        }
        asm volatile("" ::: "memory");
        wait_lgkmcnt<0>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    }
    int slot = 0, fill = kSmallMNtStages - 1;
    for (int s = s_begin; s < s_end; ++s) {
        if (issued < s_end) {
            issue_stage(fill);
            ++issued;
            fill = (fill + 1 == kSmallMNtStages) ? 0 : fill + 1;
            wait_vmcnt<kCopies * (kSmallMNtStages - 1)>();  // everything but the newest kSmallMNtStages-1 steps has landed
        } else {
            wait_vmcnt<0>();
        }
        k_step(wbase + slot * kStageBytes);
        slot = (slot + 1 == kSmallMNtStages) ? 0 : slot + 1;
        wait_lgkmcnt<0>();  // the reads of this slot are complete before a later copy refills it
    }
    if (const int k0 = ksteps * 64; NORM == 0 && k0 < K && wave == kSmallMNtWaves - 1) {
        // the last K % 64 columns, by the last wave, whose copies have all landed: zeros behind K
        const int left = K - k0 - 8 * c_chunk;
        const half8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
        half8 v[HALF_A ? 3 : 4];   // (all of them in flight before the first is looked at)
        v[0] = left > 0 ? *(const half8*)b_src0 : zero;
        v[1] = left > 0 ? *(const half8*)b_src1 : zero;
        v[2] = left > 0 ? *(const half8*)a_src0 : zero;
        if constexpr (!HALF_A) v[3] = left > 0 ? *(const half8*)a_src1 : zero;
#pragma unroll
        for (int i = 0; i < (HALF_A ? 3 : 4); ++i) {
            if ((K & 7) != 0) v[i] = first_of_chunk(v[i], left);
            *(MI355_LDS half8*)(wbase + i * 1024 + lane * 16) = v[i];
        }
        wait_lgkmcnt<0>();
        k_step(wbase);
    }

    // acc[q] is D[m = 4*(lane/16) + q][n = lane%16]; reduce the 8 partial tiles through LDS
    __syncthreads();
    MI355_LDS float* red = (MI355_LDS float*)smem;
#pragma unroll
    for (int q = 0; q < 4; ++q) red[wave * 256 + (4 * (lane >> 4) + q) * 16 + (lane & 15)] = acc[q];
    __syncthreads();
    for (int o = tid; o < 256; o += kSmallMNtWaves * 64) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < kSmallMNtWaves; ++w) sum += red[w * 256 + o];
        const int m = m0 + (o >> 4);
        if constexpr (GATE_UP) {
            if ((o & 15) < 8 && m < M) {   // column o % 16 is a gate, the one 8 further on its up
                float up = 0.f;
#pragma unroll
                for (int w = 0; w < kSmallMNtWaves; ++w) up += red[w * 256 + o + 8];
                const float sig = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-sum * 1.4426950408889634f));
                C[(long)m * ldc + 32 * (tile >> 2) + 8 * (tile & 3) + (o & 15)] = (T)(sum * sig * up);
            }
            continue;
        }
        if constexpr (EPI == kEpiRope) {
            if ((o & 15) < 8 && m < M) {
                float hi = 0.f;
#pragma unroll
                for (int w = 0; w < kSmallMNtWaves; ++w) hi += red[w * 256 + o + 8];
                store_rope_pair(epi, C, ldc, tile, m, o & 15, sum, hi);
            }
            continue;
        }
        const int n = n0 + (o & 15);
        if (m < M && n < N) {
            T v = (T)sum;
            if (R != nullptr) v = (T)((float)v + (float)R[(long)m * ldr + n]);
            C[(long)m * ldc + n] = v;
        }
    }
}

// The same product for wide weights (at least a few hundred row tiles) and K = 256 STEPS: a workgroup takes TPW
// consecutive row tiles and keeps its slice of A in registers after the first of them (a wave's K / 4 columns of the 16
// rows: 2 STEPS fragments, 128 registers at K = 4096), so from the second tile on only the weights are copied: the
// activation rows are then fetched from L2 once per TPW tiles instead of once per tile (they are as many bytes through
// the CU's memory pipeline as the weights themselves). The stream over (tile, k-step) is unrolled completely: every LDS
// offset, copy destination and wait count is an immediate, a k-step is ~18 instructions. The partial
// tiles of the four waves meet in LDS once, behind the stream (no barrier inside it).
template <typename T, bool HALF_A, int EPI, int STEPS, int TPW>
__global__ __launch_bounds__(kSmallMNtWaves * 64) void hgemm_smallm_nt_rega_kernel(const T* __restrict__ A, const T* __restrict__ B,
                                                                   T* C, const T* R, int M, int N, long lda, long ldb,
                                                                   long ldc, long ldr, int n_groups, EpilogueArgs<EPI> epi) {
    using V8 = typename Elem<T>::v8;
    constexpr bool GATE_UP = EPI == kEpiGateUp;
    constexpr int NST = kSmallMNtStages, TOTAL = TPW * STEPS;
    constexpr int kCopiesA = HALF_A ? 1 : 2;
    extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
    MI355_LDS char* smem = (MI355_LDS char*)smem_raw;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    int group = blockIdx.x;
    if (n_groups % 8 == 0) group = (blockIdx.x % 8) * (n_groups / 8) + blockIdx.x / 8;
    const int tile0 = group * TPW;
    const long kbase = (long)wave * STEPS * 64;

    // slab = 16 rows x 128 bytes; a copy instruction covers 8 rows (row lane/8, chunk position lane%8); chunk c of row r is
    // stored at position c ^ (r & 7). Lane offsets are relative to the tile's first row and the wave's first column.
    const int c_row = lane >> 3;
    const int c_chunk = (lane & 7) ^ (c_row & 7);
    const uint32_t b_voff0 = (uint32_t)((long)c_row * ldb * 2 + c_chunk * 16);
    const uint32_t b_voff1 = (uint32_t)((long)(c_row + kSmallMNtSecondRows<EPI>) * ldb * 2 + c_chunk * 16);
    const uint32_t a_voff0 = (uint32_t)((long)min(c_row, M - 1) * lda * 2 + c_chunk * 16);
    const uint32_t a_voff1 = (uint32_t)((long)min(c_row + 8, M - 1) * lda * 2 + c_chunk * 16);
    const T* a_base = A + kbase;
    const T* b_base[TPW];
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
        const int t = tile0 + i;
        b_base[i] = B + (long)smallm_nt_first_row<EPI>(t) * ldb + kbase;
    }
    const uint32_t wave_lds = (uint32_t)(uintptr_t)(smem + wave * kSmallMNtWaveBytes);

    // fragment of k-substep sub (32 deep): lane holds X[row = lane%16][k = 32*sub + 8*(lane/16) .. +7]
    const int f_row = lane & 15;
    MI355_LDS char* f_ptr[2];
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
        f_ptr[sub] = smem + wave * kSmallMNtWaveBytes + f_row * 128 + (((4 * sub + (lane >> 4)) ^ (f_row & 7)) << 4);
    MI355_LDS float* red = (MI355_LDS float*)(smem + kSmallMNtLdsBytes);   // [TPW][waves][256]

    V8 areg[STEPS][2];
    float4v acc = float4v{0.f, 0.f, 0.f, 0.f};

    auto copies_of = [](int u) { return u >= TOTAL ? 0 : u < STEPS ? 2 + kCopiesA : 2; };
    auto issue = [&](auto uc) {
        constexpr int u = decltype(uc)::value, i = u / STEPS, st = u % STEPS, slot = u % NST;
        const T* bb = b_base[i] + st * 64;   // scalar pointer arithmetic
        copy16_global_to_lds_imm<slot * kSmallMNtStageBytes>(bb, b_voff0, wave_lds);
        copy16_global_to_lds_imm<slot * kSmallMNtStageBytes + 1024>(bb, b_voff1, wave_lds);
        if constexpr (i == 0) {
            const T* ab = a_base + st * 64;
            copy16_global_to_lds_imm<slot * kSmallMNtStageBytes + 2048>(ab, a_voff0, wave_lds);
            if constexpr (!HALF_A) copy16_global_to_lds_imm<slot * kSmallMNtStageBytes + 3072>(ab, a_voff1, wave_lds);
        }
    };
    static_for<0, NST - 1>([&](auto uc) { issue(uc); });
    static_for<0, TOTAL>([&](auto uc) {
        constexpr int u = decltype(uc)::value, i = u / STEPS, st = u % STEPS, slot = u % NST;
        if constexpr (u + NST - 1 < TOTAL) issue(std::integral_constant<int, u + NST - 1>{});
        wait_vmcnt<copies_of(u + 1) + copies_of(u + 2) + copies_of(u + 3)>();   // everything up to step u has landed
        static_assert(NST == 4, "the wait above counts the three steps in flight behind step u");
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            V8 bf = Elem<T>::frag(lds_read_b128(f_ptr[sub] + slot * kSmallMNtStageBytes));
            if constexpr (i == 0) areg[st][sub] = Elem<T>::frag(lds_read_b128(f_ptr[sub] + (slot * kSmallMNtStageBytes + 2048)));
            acc = Elem<T>::mfma16(areg[st][sub], bf, acc);
        }
        wait_lgkmcnt<0>();  // the reads of this slot are complete before a later copy refills it
        if constexpr (st == STEPS - 1) {   // acc[q] is D[m = 4*(lane/16) + q][n = lane%16] of tile i
#pragma unroll
            for (int q = 0; q < 4; ++q) red[(i * kSmallMNtWaves + wave) * 256 + (4 * (lane >> 4) + q) * 16 + (lane & 15)] = acc[q];
            acc = float4v{0.f, 0.f, 0.f, 0.f};
        }
    });

    __syncthreads();
    for (int o = tid; o < TPW * 256; o += kSmallMNtWaves * 64) {
        const int i = o >> 8, e = o & 255, tile = tile0 + i;
        const MI355_LDS float* rt = red + i * kSmallMNtWaves * 256;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < kSmallMNtWaves; ++w) sum += rt[w * 256 + e];
        const int m = e >> 4;
        if constexpr (GATE_UP) {
            if ((e & 15) < 8 && m < M) {   // column e % 16 is a gate, the one 8 further on its up
                float up = 0.f;
#pragma unroll
                for (int w = 0; w < kSmallMNtWaves; ++w) up += rt[w * 256 + e + 8];
                const float sig = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-sum * 1.4426950408889634f));
                C[(long)m * ldc + 32 * (tile >> 2) + 8 * (tile & 3) + (e & 15)] = (T)(sum * sig * up);
            }
        } else if constexpr (EPI == kEpiRope) {
            if ((e & 15) < 8 && m < M) {
                float hi = 0.f;
#pragma unroll
                for (int w = 0; w < kSmallMNtWaves; ++w) hi += rt[w * 256 + e + 8];
                store_rope_pair(epi, C, ldc, tile, m, e & 15, sum, hi);
            }
        } else {
            const int n = tile * 16 + (e & 15);
            if (m < M && n < N) {
                T v = (T)sum;
                if (R != nullptr) v = (T)((float)v + (float)R[(long)m * ldr + n]);
                C[(long)m * ldc + n] = v;
            }
        }
    }
}

template <typename T, bool HALF_A, int EPI>
static hipError_t launch_smallm_nt_rega(const T* A, const T* B, T* C, const T* R, int M, int N, long lda, long ldb, long ldc,
                                        long ldr, int n_tiles, int tpw, const EpilogueArgs<EPI>& epi, hipStream_t stream) {
    static DynamicLdsOnce once4, once2;
    const int groups = n_tiles / tpw;
    if (tpw == 4) {
        constexpr int lds = kSmallMNtLdsBytes + 4 * kSmallMNtWaves * 1024;
        auto kern = hgemm_smallm_nt_rega_kernel<T, HALF_A, EPI, 16, 4>;
        if (hipError_t e = once4.ensure(reinterpret_cast<const void*>(kern), lds); e != hipSuccess) return e;
        kern<<<dim3(groups), dim3(kSmallMNtWaves * 64), lds, stream>>>(A, B, C, R, M, N, lda, ldb, ldc, ldr, groups, epi);
    } else {
        constexpr int lds = kSmallMNtLdsBytes + 2 * kSmallMNtWaves * 1024;
        auto kern = hgemm_smallm_nt_rega_kernel<T, HALF_A, EPI, 16, 2>;
        if (hipError_t e = once2.ensure(reinterpret_cast<const void*>(kern), lds); e != hipSuccess) return e;
        kern<<<dim3(groups), dim3(kSmallMNtWaves * 64), lds, stream>>>(A, B, C, R, M, N, lda, ldb, ldc, ldr, groups, epi);
    }
    return hipGetLastError();
}

template <typename T, bool HALF_A, int EPI>
static hipError_t launch_smallm_nt_half(const T* A, const T* B, T* C, const T* R, int M, int N, int K, long lda, long ldb, long ldc,
                                        long ldr, int tpw, const EpilogueArgs<EPI>& epi, hipStream_t stream) {
    static DynamicLdsOnce once;
    const int n_tiles = (N + 15) / 16;
    if (tpw > 0) return launch_smallm_nt_rega<T, HALF_A, EPI>(A, B, C, R, M, N, lda, ldb, ldc, ldr, n_tiles, tpw, epi, stream);
    auto kern = hgemm_smallm_nt_kernel<T, HALF_A, EPI>;
    if (hipError_t e = once.ensure(reinterpret_cast<const void*>(kern), kSmallMNtLdsBytes); e != hipSuccess) return e;
    kern<<<dim3(n_tiles, (M + 15) / 16), dim3(kSmallMNtWaves * 64), kSmallMNtLdsBytes, stream>>>(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, n_tiles, epi,
                                                                                                 nullptr, 0.f);
    return hipGetLastError();
}

// EPI kEpiGateUp: silu(A gate^T) * (A up^T) for up to 16 rows: N counts the rows of B ([32 gate | 32 up] groups, a multiple of
// 64), C is [M, N / 2]. kEpiRope: up to 64 rows, N whole heads.
template <typename T, int EPI = kEpiPlain>
static hipError_t launch_smallm_nt(const T* A, const T* B, T* C, const T* R, int M, int N, int K, long lda, long ldb,
                                   long ldc, long ldr, hipStream_t stream, const EpilogueArgs<EPI>& epi = {}) {
    const int tpw = N % 16 == 0 ? smallm_nt_rega_tpw(M, N / 16, K, lda, ldb) : 0;
    if (M <= 8) return launch_smallm_nt_half<T, true, EPI>(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, tpw, epi, stream);
    return launch_smallm_nt_half<T, false, EPI>(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, tpw, epi, stream);
}

template <typename T, int EPI>
static hipError_t launch_smallm_nt_norm(const T* A, const T* norm_weight, float eps, const T* B, T* C, int M, int N, int K, long lda, long ldb,
                                        long ldc, hipStream_t stream, const EpilogueArgs<EPI>& epi) {
    const int n_tiles = N / 16;
    const auto launch = [&](auto rows) -> hipError_t {
        static DynamicLdsOnce once;
        auto kern = hgemm_smallm_nt_kernel<T, true, EPI, decltype(rows)::value>;
        if (hipError_t e = once.ensure(reinterpret_cast<const void*>(kern), kNormLdsMax); e != hipSuccess) return e;
        kern<<<dim3(n_tiles), dim3(kSmallMNtWaves * 64), smallm_nt_norm_lds(M, K), stream>>>(A, B, C, nullptr, M, N, K, lda, ldb, ldc, 0, n_tiles, epi,
                                                                                              norm_weight, eps);
        return hipGetLastError();
    };
    switch (smallm_nt_norm_rows(M)) {
        case 1: return launch(std::integral_constant<int, 1>{});
        case 2: return launch(std::integral_constant<int, 2>{});
        case 4: return launch(std::integral_constant<int, 4>{});
        default: return launch(std::integral_constant<int, 8>{});
    }
}

// One workgroup per tile, so that a CU is given back after every tile. (256 workgroups that walk the tiles, and request the next
// tile's operands in front of the stores of the last, gain 0-1 % of a product alone: 8192^3 NN 805.2 us against 805.8 on one card, 781
// against 787 on another. With one CU held by a kernel of another stream the workgroup left over begins its walk when the others end
// theirs, 8192^3 1.66 times its time alone against 1.10, 8192 x 28672 x 4096 gate/up 1.80 against 1.02; an RMSNorm of 8 rows on another
// stream waits for the whole product, 831 us against 220.)
template <typename T, bool A_KC, bool B_KC, int BM, int BN, int WM, int WN, int EPI = 0, bool RAGGED = false, int STAGES = 0, int PER_CU = 1>
static hipError_t launch_main(const T* A, const T* B, T* C, const T* R, int M, int N, int K, long lda, long ldb,
                              long ldc, long ldr, hipStream_t stream) {
    using Cfg = MainCfg<A_KC, B_KC, BM, BN, WM, WN, STAGES>;
    auto kern = hgemm_main_kernel<T, A_KC, B_KC, BM, BN, WM, WN, EPI, RAGGED, STAGES, PER_CU>;
    static DynamicLdsOnce lds_once;
    if (hipError_t e = lds_once.ensure(reinterpret_cast<const void*>(kern), Cfg::LDS_BYTES); e != hipSuccess) return e;
    const long nblocks = (long)((M + BM - 1) / BM) * ((N + BN - 1) / BN);
    if (nblocks > 0x7fffffffL) return hipErrorInvalidValue;
    const int blocks = (int)nblocks;
    MI355_TL(timeline_hgemm_reader = &read_hgemm_stamps;)
    kern<<<dim3(blocks), dim3(Cfg::NTHREADS), Cfg::LDS_BYTES, stream>>>(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, nullptr, nullptr, 1);
    return hipGetLastError();
}

// hipErrorStreamCaptureUnsupported / hipErrorOutOfMemory: no workspace to be had, the caller takes another kernel.
// own_merge: the partial tiles are merged by hgemm_merge_kernel instead of the last workgroup of each tile.
template <typename T, bool A_KC, bool B_KC, int BM, int BN, int WM, int WN, int STAGES = 0, int PER_CU = 1>
static hipError_t launch_split_k(const T* A, const T* B, T* C, const T* R, int M, int N, int K, long lda, long ldb, long ldc,
                                 long ldr, int splits, bool own_merge, hipStream_t stream) {
    using Cfg = MainCfg<A_KC, B_KC, BM, BN, WM, WN, STAGES>;
    auto kern = hgemm_main_kernel<T, A_KC, B_KC, BM, BN, WM, WN, 0, true, STAGES, PER_CU, true>;
    static DynamicLdsOnce lds_once;
    if (hipError_t e = lds_once.ensure(reinterpret_cast<const void*>(kern), Cfg::LDS_BYTES); e != hipSuccess) return e;
    if (kOwnMergeOnly<BM, BN>) own_merge = true;
    const long tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN, tiles = tiles_m * tiles_n;
    if (!own_merge && tiles * sizeof(unsigned) > kSplitKCounterBytes) return hipErrorOutOfMemory;
    const size_t bytes = kSplitKCounterBytes + (size_t)tiles * splits * BM * BN * 4;
    char* ws = nullptr;
    std::unique_lock<std::mutex> order;   // the launches below follow one another on the stream
    if (hipError_t e = split_k_workspace(bytes, stream, &ws, &order); e != hipSuccess) return e;
    float* part = reinterpret_cast<float*>(ws + kSplitKCounterBytes);
    MI355_TL(timeline_hgemm_reader = &read_hgemm_stamps;)
    kern<<<dim3((unsigned)tiles, (unsigned)splits), dim3(Cfg::NTHREADS), Cfg::LDS_BYTES, stream>>>(
        A, B, C, R, M, N, K, lda, ldb, ldc, ldr, part, own_merge ? nullptr : reinterpret_cast<unsigned*>(ws), splits);
    if (own_merge) {
        const long mp = tiles_m * BM, np = tiles_n * BN, threads = (long)M * (np / 8);
        hgemm_merge_kernel<T><<<dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream>>>(part, C, R, M, N, mp, np, ldc, ldr, splits);
    }
    return hipGetLastError();
}

// see mi355_internal_hgemm_variant
static KernelChoice pinned_kernel(int variant, int K) {
    KernelChoice k;
    k.shape = variant & 15;
    k.splits = std::min((variant >> 4) & 0xff, (K + 63) / 64);   // a range is at least one K tile: an empty one would copy a whole tile from behind K
    if (k.splits < 1) k.splits = 1;
    k.own_merge = (variant >> 12) != 0;
    if (k.shape == kSmallM && k.splits > 1) std::swap(k.splits, k.wide_ranges);
    return k;
}
// hipErrorNotSupported: no such kernel for this layout
template <typename T, bool A_KC, bool B_KC>
static hipError_t run_kernel(const KernelChoice& k, const T* A, const T* B, T* C, const T* R, int M, int N, int K, long lda, long ldb,
                             long ldc, long ldr, bool c_aligned, hipStream_t stream) {
#define MI355_ARGS A, B, C, R, M, N, K, lda, ldb, ldc, ldr
    if constexpr (!B_KC)
        if (k.shape == kSmallM && k.wide_ranges > 1) return launch_smallm_wide<T, A_KC>(MI355_ARGS, k.wide_ranges, stream);
    if (k.splits > 1) {
        switch (k.shape) {
            case kTile128x128: return launch_split_k<T, A_KC, B_KC, 128, 128, 2, 2>(MI355_ARGS, k.splits, k.own_merge, stream);
            case kTileHalf:
                if constexpr (A_KC && B_KC) return launch_split_k<T, A_KC, B_KC, 128, 64, 2, 2>(MI355_ARGS, k.splits, k.own_merge, stream);
                else return launch_split_k<T, A_KC, B_KC, 64, 128, 1, 4>(MI355_ARGS, k.splits, k.own_merge, stream);
            case kTile64x64: return launch_split_k<T, A_KC, B_KC, 64, 64, 2, 2, 4, 2>(MI355_ARGS, k.splits, k.own_merge, stream);
            case kTile128x256: return launch_split_k<T, A_KC, B_KC, 128, 256, 2, 4>(MI355_ARGS, k.splits, k.own_merge, stream);
            case kTile256x128: return launch_split_k<T, A_KC, B_KC, 256, 128, 4, 2>(MI355_ARGS, k.splits, k.own_merge, stream);
            case kTile256x256: return launch_split_k<T, A_KC, B_KC, 256, 256, 2, 4>(MI355_ARGS, k.splits, k.own_merge, stream);
            case kTile32x64:
                if constexpr (A_KC) return launch_split_k<T, A_KC, B_KC, 32, 64, 2, 2, 4, 2>(MI355_ARGS, k.splits, k.own_merge, stream);
                else return hipErrorNotSupported;
            default: return hipErrorNotSupported;
        }
    }
    const auto whole = [&](int bm, int bn) { return c_aligned && M % bm == 0 && N % bn == 0 && K % 8 == 0; };
    switch (k.shape) {
        case kTile256x256:
            if (whole(256, 256)) return launch_main<T, A_KC, B_KC, 256, 256, 2, 4>(MI355_ARGS, stream);
            return launch_main<T, A_KC, B_KC, 256, 256, 2, 4, 0, true>(MI355_ARGS, stream);
        case kTile128x128:
            if (whole(128, 128)) return launch_main<T, A_KC, B_KC, 128, 128, 2, 2>(MI355_ARGS, stream);
            return launch_main<T, A_KC, B_KC, 128, 128, 2, 2, 0, true>(MI355_ARGS, stream);
        case kTileHalf:
            if constexpr (A_KC && B_KC) {
                if (whole(128, 64)) return launch_main<T, A_KC, B_KC, 128, 64, 2, 2>(MI355_ARGS, stream);
                return launch_main<T, A_KC, B_KC, 128, 64, 2, 2, 0, true>(MI355_ARGS, stream);
            } else {
                if (whole(64, 128)) return launch_main<T, A_KC, B_KC, 64, 128, 1, 4>(MI355_ARGS, stream);
                return launch_main<T, A_KC, B_KC, 64, 128, 1, 4, 0, true>(MI355_ARGS, stream);
            }
        case kTile64x64:
            if (whole(64, 64)) return launch_main<T, A_KC, B_KC, 64, 64, 2, 2, 0, false, 4, 2>(MI355_ARGS, stream);
            return launch_main<T, A_KC, B_KC, 64, 64, 2, 2, 0, true, 4, 2>(MI355_ARGS, stream);
        case kTile128x256:
            if (whole(128, 256)) return launch_main<T, A_KC, B_KC, 128, 256, 2, 4>(MI355_ARGS, stream);
            return launch_main<T, A_KC, B_KC, 128, 256, 2, 4, 0, true>(MI355_ARGS, stream);
        case kTile256x128:
            if (whole(256, 128)) return launch_main<T, A_KC, B_KC, 256, 128, 4, 2>(MI355_ARGS, stream);
            return launch_main<T, A_KC, B_KC, 256, 128, 4, 2, 0, true>(MI355_ARGS, stream);
        case kTile32x64:
            if constexpr (A_KC) return launch_main<T, A_KC, B_KC, 32, 64, 2, 2, 0, true, 8>(MI355_ARGS, stream);
            else return hipErrorNotSupported;
        case kDeepRing:
            return launch_main<T, A_KC, B_KC, 64, 64, 2, 2, 0, true>(MI355_ARGS, stream);
        case kSmallM:
            if constexpr (!B_KC) return launch_smallm_nn<T, A_KC>(MI355_ARGS, stream);
            else if constexpr (A_KC) return launch_smallm_nt<T>(MI355_ARGS, stream);
            else return hipErrorNotSupported;
        default: return hipErrorNotSupported;
    }
#undef MI355_ARGS
}

template <typename T, bool A_KC, bool B_KC>
static hipError_t launch_layout(const T* A, const T* B, T* C, const T* R, int M, int N, int K, long lda, long ldb,
                                long ldc, long ldr, int variant, hipStream_t stream) {
    // the copies of the fast kernels move 16 bytes into LDS: the operands' rows must be 16-byte aligned. C and the residual
    // may lie anywhere; the kernels that assume whole tiles also assume aligned rows of C (c_aligned).
    const bool ab_aligned = (reinterpret_cast<uintptr_t>(A) % 16 == 0) && (reinterpret_cast<uintptr_t>(B) % 16 == 0) &&
                            (lda % 8 == 0) && (ldb % 8 == 0);
    const bool c_aligned = (reinterpret_cast<uintptr_t>(C) % 16 == 0) && (ldc % 8 == 0) &&
                           (reinterpret_cast<uintptr_t>(R) % 16 == 0) && (ldr % 8 == 0);
    // Any K: where it ends inside a 16-byte chunk of a row, the kernels put zeros in the place of what follows in that chunk.
    // Any N: an operand stored [K,N] is copied in 16-byte chunks of its rows, and the chunk that straddles N ends in the padding
    // a leading dimension of a multiple of 8 leaves (what it holds only reaches columns that are never stored).
    if (ab_aligned) {
        // the tiled kernels address a tile with 32-bit byte offsets: up to 256 rows of lda (ldb) elements
        const bool tiles_ok = lda < (1L << 22) && ldb < (1L << 22);
        const bool whole_lines = ldb % 64 == 0;
        KernelChoice pick = variant > 0 && (A_KC || (variant & 15) != kTile32x64) && (tiles_ok || (variant & 15) == kSmallM) ? pinned_kernel(variant, K) : choose_kernel(M, N, K, A_KC, B_KC, tiles_ok, true, whole_lines);
        for (;;) {
            const hipError_t e = run_kernel<T, A_KC, B_KC>(pick, A, B, C, R, M, N, K, lda, ldb, ldc, ldr, c_aligned, stream);
            // no workspace to be had (the stream is being captured and has none yet): the best kernel without split-K
            if ((pick.splits <= 1 && pick.wide_ranges <= 1) || variant > 0 || (e != hipErrorStreamCaptureUnsupported && e != hipErrorOutOfMemory)) {
                if (e != hipErrorNotSupported) return e;
                break;
            }
            (void)hipGetLastError();
            pick = choose_kernel(M, N, K, A_KC, B_KC, tiles_ok, false, whole_lines);
        }
    }
    return gemm_direct_dispatch(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, A_KC ? (B_KC ? MI355_GEMM_NT : MI355_GEMM_NN) : MI355_GEMM_TN,
                                std::is_same<T, bf16_t>::value ? MI355_DTYPE_BF16 : MI355_DTYPE_FP16, 0, stream);
}

// Product with the gate/up epilogue (EPI = 1): N counts the columns of op(B) (twice those of C). Operands that are not
// 16-byte aligned, K that is not a multiple of 64 or N that is not a multiple of 64 report hipErrorNotSupported and the
// caller runs the product and mi355_silu_mul separately.
template <typename T, bool A_KC, bool B_KC>
static hipError_t launch_silu_mul(const T* A, const T* B, T* C, int M, int N, int K, long lda, long ldb,
                                  long ldc, int variant, hipStream_t stream) {
    const bool aligned = (reinterpret_cast<uintptr_t>(A) % 16 == 0) && (reinterpret_cast<uintptr_t>(B) % 16 == 0) &&
                         (reinterpret_cast<uintptr_t>(C) % 16 == 0) && (lda % 8 == 0) && (ldb % 8 == 0) && (ldc % 8 == 0);
    // N = columns of op(B); gate/up pairs are 64 columns wide. Few rows are better served by the small-M product.
    if (!aligned || K % 64 != 0 || K < 64 || N % 64 != 0 || lda >= (1L << 22) || ldb >= (1L << 22)) return hipErrorNotSupported;
    if constexpr (A_KC && B_KC) {   // generation step: the split-K small-M kernel with the same epilogue
        if (M <= 16 && (variant == 0 || variant == kSmallM)) return launch_smallm_nt<T, kEpiGateUp>(A, B, C, nullptr, M, N, K, lda, ldb, ldc, 0, stream);
    }
    // More rows: the tile shape by the same model as the plain product's. On 64x64 tiles four waves lie side by side along M,
    // so that every wave holds the gate and the up columns of its rows.
#define MI355_ARGS A, B, C, nullptr, M, N, K, lda, ldb, ldc, 0
    switch (variant > 0 ? variant : choose_kernel(M, N, K, A_KC, B_KC, true, false, ldb % 64 == 0, true).shape) {
        case kTile256x256:
            if (M % 256 == 0 && N % 256 == 0) return launch_main<T, A_KC, B_KC, 256, 256, 2, 4, 1>(MI355_ARGS, stream);
            return launch_main<T, A_KC, B_KC, 256, 256, 2, 4, 1, true>(MI355_ARGS, stream);
        case kTile128x256: return launch_main<T, A_KC, B_KC, 128, 256, 2, 4, 1, true>(MI355_ARGS, stream);
        case kTile256x128: return launch_main<T, A_KC, B_KC, 256, 128, 4, 2, 1, true>(MI355_ARGS, stream);
        case kTile64x64: return launch_main<T, A_KC, B_KC, 64, 64, 4, 1, 1, true, 4, 2>(MI355_ARGS, stream);
        case kDeepRing: return launch_main<T, A_KC, B_KC, 64, 64, 4, 1, 1, true>(MI355_ARGS, stream);
        default:
            if (M % 128 == 0 && N % 128 == 0) return launch_main<T, A_KC, B_KC, 128, 128, 2, 2, 1>(MI355_ARGS, stream);
            return launch_main<T, A_KC, B_KC, 128, 128, 2, 2, 1, true>(MI355_ARGS, stream);
    }
#undef MI355_ARGS
}

// The first two products of a generation step's layer, few enough rows for the small-M kernel of layout NT, with what stands
// around them: the RMSNorm of their rows in front (norm.weight != nullptr), rotary embedding and the way into the KV cache behind
// the QKV projection. hipErrorNotSupported: no such kernel for this call, nothing was launched.
// Every workgroup normalises the rows for itself (~0.2 us a row, hidden behind the first weights in part), with two workgroups and
// their rows on a CU at most, so a product of many workgroups pays for it once per round of 512, and for more than two rows that
// exceeds the launch it saves where the rows are long. us, weights from HBM, norm on its own / in the product: gate/up 8 rows 1536 x
// 4096 9.7 / 8.7 (1 round), x 8960 15.6 / 18.2 (3), 2048 x 7168 16.2 / 15.5 (2), x 16384 28.8 / 31.0 (4), 2560 x 4096 12.8 / 11.6 (1), x 6912
// 19.1 / 19.5 (2); 4 rows 2560 x 10240 23.1 / 22.2 (3), 3072 x 16384 38.1 / 37.3 (4), 3584 x 18944 48.7 / 48.8 (5), 4096 x 11008 35.1 / 34.0
// (3), x 14336 41.7 / 43.2 (4); 1 and 2 rows gain 0 - 3 us at any width (4096 x 14336 41.6 / 41.7, 6144 x 24576 100.6 / 98.8, 8192 x 28672,
// one row, 152.4 / 151.0). Over more than one round the kernel that keeps the rows in registers is the better one where it
// applies (4096 x 8192, 4 rows, 27.6 / 28.4, 1 row 27.3 / 27.6). QKV projections are one or two rounds: 4096 x 6144 4 rows 14.1 / 12.5, 1024 x
// 1536 8 rows 6.0 / 5.5, also where the choice by shape would take another kernel than the small-M one: 1024 x 16384 8 rows 14.3 / 14.0,
// 1 row 13.8 / 8.2, 11264 x 1280 20.9 / 13.1.
static bool norm_fits(const NormPrologue& norm, int M, int N, int K) {
    if (M > 8 || K < 1024 || K % 512 != 0 || smallm_nt_norm_lds(M, K) > kNormLdsMax - 1024 || reinterpret_cast<uintptr_t>(norm.weight) % 16 != 0)
        return false;
    const int rows = smallm_nt_norm_rows(M);
    const long rounds = (N / 16 + 511) / 512;
    if (rounds > 1 && smallm_nt_rega_tpw(M, N / 16, K, K, K) > 0) return false;
    return rows <= 2 || rounds * K <= (rows == 4 ? 12288 : 4096);
}

template <typename T>
hipError_t gemm_step_qkv(const void* x, const NormPrologue& norm, const void* w, void* qkv, int M, int N, int K, long ldx, long ldb, long ldc,
                         const RopeEpilogue& rope, hipStream_t stream) {
    const T *A = static_cast<const T*>(x), *B = static_cast<const T*>(w);
    T* C = static_cast<T*>(qkv);
    const bool aligned = reinterpret_cast<uintptr_t>(A) % 16 == 0 && reinterpret_cast<uintptr_t>(B) % 16 == 0 && ldx % 8 == 0 && ldb % 8 == 0;
    if (!aligned || M > 64 || N % 128 != 0 || ldx >= (1L << 22) || ldb >= (1L << 22)) return hipErrorNotSupported;
    if (norm.weight != nullptr) {
        if (!norm_fits(norm, M, N, K)) return hipErrorNotSupported;
        return launch_smallm_nt_norm<T, kEpiRope>(A, static_cast<const T*>(norm.weight), norm.eps, B, C, M, N, K, ldx, ldb, ldc, stream, rope);
    }
    if (choose_kernel(M, N, K, true, true, true, true, ldb % 64 == 0).shape != kSmallM) return hipErrorNotSupported;
    return launch_smallm_nt<T, kEpiRope>(A, B, C, nullptr, M, N, K, ldx, ldb, ldc, 0, stream, rope);
}

template <typename T>
hipError_t gemm_step_gate_up(const void* x, const NormPrologue& norm, const void* w, void* out, int M, int N, int K, long ldx, long ldb, long ldc,
                             hipStream_t stream) {
    const T *A = static_cast<const T*>(x), *B = static_cast<const T*>(w);
    const bool aligned = reinterpret_cast<uintptr_t>(A) % 16 == 0 && reinterpret_cast<uintptr_t>(B) % 16 == 0 && ldx % 8 == 0 && ldb % 8 == 0;
    if (!aligned || N % 64 != 0 || !norm_fits(norm, M, N, K)) return hipErrorNotSupported;
    return launch_smallm_nt_norm<T, kEpiGateUp>(A, static_cast<const T*>(norm.weight), norm.eps, B, static_cast<T*>(out), M, N, K, ldx, ldb, ldc,
                                                stream, {});
}

// One translation unit per element type and layout (the build compiles the six side by side): MI355_HGEMM_T and
// MI355_HGEMM_LAYOUT select it; without them everything is instantiated here.
template <typename T, int LAYOUT>
hipError_t gemm_layout(const void* A, const void* B, void* C, const void* R, int M, int N, int K, long lda, long ldb, long ldc,
                       long ldr, int variant, hipStream_t stream) {
    return launch_layout<T, LAYOUT != MI355_GEMM_TN, LAYOUT == MI355_GEMM_NT>(
        static_cast<const T*>(A), static_cast<const T*>(B), static_cast<T*>(C), static_cast<const T*>(R), M, N, K, lda, ldb, ldc, ldr,
        variant, stream);
}
template <typename T, int LAYOUT>
hipError_t gemm_silu_mul_layout(const void* A, const void* B, void* C, int M, int N2, int K, long lda, long ldb, long ldc,
                                int variant, hipStream_t stream) {
    if constexpr (LAYOUT == MI355_GEMM_TN) return hipErrorNotSupported;
    else return launch_silu_mul<T, true, LAYOUT == MI355_GEMM_NT>(static_cast<const T*>(A), static_cast<const T*>(B), static_cast<T*>(C),
                                                                  M, N2, K, lda, ldb, ldc, variant, stream);
}
#define MI355_HGEMM_INSTANTIATE(T, LAYOUT)                                                                                     \
    template hipError_t gemm_layout<T, LAYOUT>(const void*, const void*, void*, const void*, int, int, int, long, long, long,  \
                                               long, int, hipStream_t);                                                        \
    template hipError_t gemm_silu_mul_layout<T, LAYOUT>(const void*, const void*, void*, int, int, int, long, long, long, int, hipStream_t);
#define MI355_HGEMM_INSTANTIATE_STEP(T)                                                                                        \
    template hipError_t gemm_step_qkv<T>(const void*, const NormPrologue&, const void*, void*, int, int, int, long, long, long, \
                                         const RopeEpilogue&, hipStream_t);                                                    \
    template hipError_t gemm_step_gate_up<T>(const void*, const NormPrologue&, const void*, void*, int, int, int, long, long, long, hipStream_t);
#ifdef MI355_HGEMM_T
MI355_HGEMM_INSTANTIATE(MI355_HGEMM_T, MI355_HGEMM_LAYOUT)
#ifdef MI355_HGEMM_STEP
MI355_HGEMM_INSTANTIATE_STEP(MI355_HGEMM_T)
#endif
#else
MI355_HGEMM_INSTANTIATE_STEP(half_t)
MI355_HGEMM_INSTANTIATE_STEP(bf16_t)
MI355_HGEMM_INSTANTIATE(half_t, MI355_GEMM_NN)
MI355_HGEMM_INSTANTIATE(half_t, MI355_GEMM_NT)
MI355_HGEMM_INSTANTIATE(half_t, MI355_GEMM_TN)
MI355_HGEMM_INSTANTIATE(bf16_t, MI355_GEMM_NN)
MI355_HGEMM_INSTANTIATE(bf16_t, MI355_GEMM_NT)
MI355_HGEMM_INSTANTIATE(bf16_t, MI355_GEMM_TN)
#endif

}  // namespace mi355
