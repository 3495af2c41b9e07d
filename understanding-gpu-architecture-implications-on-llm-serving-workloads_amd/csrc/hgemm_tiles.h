// What the tiled GEMM kernels share: how an operand tile lies in LDS and how its fragments are read, how a wave stores its
// sub-tile of C, and how partial tiles of ranges of K are merged.
#pragma once
#include <type_traits>
#include "mi355_common.h"

namespace mi355 {

// f(std::integral_constant<int, I>) for I = BEGIN .. END-1, unrolled at compile time
template <int BEGIN, int END, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (BEGIN < END) {
        f(std::integral_constant<int, BEGIN>{});
        static_for<BEGIN + 1, END>(f);
    }
}

// ---------------------------------------------------------------------------------------------------------
// LDS tile descriptions
// ---------------------------------------------------------------------------------------------------------

// Operand tile whose K index is contiguous in memory: LDS holds [ROWS][BK] halfs, row = M (or N) index.
// 16-byte chunk c of row r lives at chunk position c ^ swz(r).
template <int ROWS, int BK, int NWAVES>
struct KContigTile {
    static constexpr int kChunksPerRow = BK / 8;
    static constexpr int kRowBytes = BK * 2;
    static constexpr int kRowsPerInst = 64 / kChunksPerRow;
    static constexpr int kRowsPerPass = kRowsPerInst * NWAVES;
    static constexpr int kInsts = ROWS / kRowsPerPass;
    static constexpr int kBytes = ROWS * kRowBytes;
    static_assert(ROWS % kRowsPerPass == 0, "tile rows must be a multiple of one pass of the workgroup");
    static_assert(BK == 64, "swizzle below is written for 128-byte rows");

    // A fragment read (ds_read_b128) has lane l at row l % 16, chunk c0 + l / 16. Rows of equal parity share the same
    // half of the 256-byte bank window, so their chunk positions must differ: over 16 consecutive lanes (16 rows, one
    // chunk), and over the lanes l and l + 32 that the hardware serves together (8 rows, chunks c and c + 2, i.e. c ^ 2).
    // Bits 0 and 2 of the XOR value tell the 4 rows of one parity inside an 8-row group apart, bit 1 the two groups.
    __device__ static __forceinline__ int swz(int row) {
        return ((row >> 1) & 1) | (((row >> 2) & 1) << 2) | (((row >> 3) & 1) << 1);
    }

    // element offset (in halfs, relative to the tile origin in global memory) of this lane's first copy
    __device__ static __forceinline__ long first_copy_offset(int wave, int lane, long ld) {
        int row = wave * kRowsPerInst + lane / kChunksPerRow;
        int chunk = (lane % kChunksPerRow) ^ swz(row);
        return (long)row * ld + chunk * 8;
    }
    __device__ static __forceinline__ long copy_stride(long ld) { return (long)kRowsPerPass * ld; }
    __device__ static __forceinline__ long ktile_stride(long /*ld*/) { return BK; }
    __device__ static __forceinline__ int lds_inst_offset(int inst, int wave) { return (inst * NWAVES + wave) * 1024; }

    // byte offset inside the tile of this lane's 16 bytes of the fragment (16 rows x 32 k) for k-substep kk, first
    // row row0 (a multiple of 16): lane l holds k = 32 kk + 8 (l / 16) .. +7 of row l % 16
    __device__ static __forceinline__ int frag_offset(int row0, int kk, int lane) {
        int row = row0 + (lane & 15);
        int chunk = (kk * 4 + (lane >> 4)) ^ swz(row);
        return row * kRowBytes + chunk * 16;
    }
};

// Operand tile whose M/N index is contiguous in memory: LDS holds [BK][COLS] halfs, row = K index.
template <int COLS, int BK, int NWAVES>
struct MNContigTile {
    static constexpr int kChunksPerRow = COLS / 8;
    static constexpr int kRowBytes = COLS * 2;
    static constexpr int kRowsPerInst = 64 / kChunksPerRow;
    static constexpr int kRowsPerPass = kRowsPerInst * NWAVES;
    static constexpr int kInsts = BK / kRowsPerPass;
    static constexpr int kBytes = BK * kRowBytes;
    static_assert(COLS == 256 || COLS == 128 || COLS == 64, "the swizzles below are written for these row lengths");
    static_assert(kRowsPerPass % 16 == 0, "copy i of a lane is 16 rows or a multiple further down: same swizzle for all i");
    static_assert(BK % kRowsPerPass == 0, "tile depth must be a multiple of one pass of the workgroup");

    // A transposing read touches, per 16 lanes, 4 k-rows x 32 bytes (two neighbouring chunks); lanes 0..31 of a
    // fragment read cover rows {0..3} and {8..11} (+ a multiple of 4 that does not change what follows). XOR-ing the
    // chunk index with an even number that differs for those 8 rows keeps their 8 chunk pairs on distinct banks.
    // Rows of 128 bytes (COLS == 64) fill only half of the 256-byte bank window: rows of equal parity share a half, so
    // it is the 4 rows of one parity among those 8 that need distinct chunk pairs (bits 1 and 3 of the row tell them apart).
    __device__ static __forceinline__ int swz(int row) {
        if constexpr (COLS == 64) return (((row >> 1) & 1) | (((row >> 3) & 1) << 1)) << 1;
        else return ((row & 3) | (((row >> 3) & 1) << 2)) << 1;
    }
    __device__ static __forceinline__ long first_copy_offset(int wave, int lane, long ld) {
        int row = wave * kRowsPerInst + lane / kChunksPerRow;
        int chunk = (lane % kChunksPerRow) ^ swz(row);
        return (long)row * ld + chunk * 8;
    }
    __device__ static __forceinline__ long copy_stride(long ld) { return (long)kRowsPerPass * ld; }
    __device__ static __forceinline__ long ktile_stride(long ld) { return (long)BK * ld; }
    __device__ static __forceinline__ int lds_inst_offset(int inst, int wave) { return (inst * NWAVES + wave) * 1024; }

    // byte offset of this lane's transposing read for the fragment (32 k x 16 cols) whose first column is col0 (a
    // multiple of 16): group g = lane / 16 reads k rows 8g .. 8g+3, input lane j of the group supplies the 4 columns
    // 4 (j % 4) .. +3 of row j / 4. Add (kk*32 + 4*t) * kRowBytes for substep kk and half t (neither changes swz).
    __device__ static __forceinline__ int frag_offset(int col0, int lane) {
        int j = lane & 15;
        int row = 8 * (lane >> 4) + (j >> 2);
        int chunk = (col0 >> 3) + ((j & 3) >> 1);
        return row * kRowBytes + ((chunk ^ swz(row)) << 4) + (j & 1) * 8;
    }
};

// the first `left` of the 8 elements of a 16-byte chunk, zeros behind them
__device__ __forceinline__ half8 first_of_chunk(half8 chunk, int left) {
    int4v v = __builtin_bit_cast(int4v, chunk);
#pragma unroll
    for (int w = 0; w < 4; ++w) v[w] = 2 * w >= left ? 0 : 2 * w + 1 == left ? v[w] & 0xffff : v[w];
    return __builtin_bit_cast(half8, v);
}

// Epilogue of the tiled kernels for one wave's sub-tile of TM x TN blocks of 16x16 (first row row0, first stored column
// col0, of a C with NC columns). A lane holds C[m][n .. n+3] for m = l%16, n = 4*(l/16) of every block. Storing that
// directly would write 8-byte pieces of 16 different rows per instruction (partial cache lines, read-modify-write in
// the memory system), so the wave first parks its sub-tile in its own slice of LDS (cst; fp16, 16-byte chunks
// XOR-swizzled by row) and then stores whole rows: every store instruction writes complete 128-byte lines.
// EPI == 1: the wave's columns come in groups of [32 gate | 32 up]; output block jo takes its gate from block
// 4 (jo / 2) + jo % 2 and its up from two blocks further.
template <typename T, int TM, int TN, int EPI, bool RAGGED>
__device__ __forceinline__ void store_wave_tile(const float4v (&acc)[TM][TN], MI355_LDS char* cst, T* C, const T* R, long row0,
                                                long col0, int M, int NC, long ldc, long ldr, int lane) {
    using V8 = typename Elem<T>::v8;
    using V4 = typename Elem<T>::v4;
    static_assert(EPI == 0 || TN % 4 == 0, "the gate/up epilogue pairs column blocks 32 columns apart");
    constexpr int TNO = EPI == 1 ? TN / 2 : TN;   // column blocks a wave stores
    constexpr int kRowHalfs = TNO * 16;           // width of the stored wave sub-tile
    constexpr int kRowBytesC = kRowHalfs * 2;
    constexpr int kChunksC = kRowBytesC / 16;     // 16-byte chunks per row (4, 8 or 16)
    constexpr int kRowsPerStore = 64 / kChunksC;  // rows covered by one store instruction
    constexpr int kSwzC = kChunksC < 8 ? kChunksC - 1 : 7;
    {
        const int r = lane & 15;
        const int g = lane >> 4;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int row = i * 16 + r;
#pragma unroll
            for (int jo = 0; jo < TNO; ++jo) {
                V4 v;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if constexpr (EPI == 1) {
                        const int gj = (jo / 2) * 4 + (jo % 2);
                        const float gt = acc[i][gj][q];
                        const float sig = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-gt * 1.4426950408889634f));
                        v[q] = (T)(gt * sig * acc[i][gj + 2][q]);
                    } else {
                        v[q] = (T)acc[i][jo][q];
                    }
                }
                const int chunk = (2 * jo + (g >> 1)) ^ (row & kSwzC);
                *(MI355_LDS V4*)(cst + row * kRowBytesC + chunk * 16 + (g & 1) * 8) = v;
            }
        }
    }
    // only this wave reads what it wrote: no workgroup barrier needed, the LDS operations of a wave complete in order
    {
        const int rr = lane / kChunksC;
        const int cc = lane % kChunksC;
        T* cbase = C + row0 * ldc + col0 + cc * 8;
        const long rows_left = M - row0;   // RAGGED: rows and columns that exist
        const long cols_left = NC - (col0 + cc * 8);   // of this lane's 8
        const T* rbase = R + row0 * ldr + col0 + cc * 8;
#pragma unroll
        for (int it = 0; it < TM * 16 / kRowsPerStore; ++it) {
            const int row = it * kRowsPerStore + rr;
            V8 v = *(MI355_LDS const V8*)(cst + row * kRowBytesC + ((cc ^ (row & kSwzC)) << 4));
            if constexpr (!RAGGED) {
                if (R != nullptr) {
                    const V8 r = *(const V8*)(rbase + (long)row * ldr);
#pragma unroll
                    for (int j = 0; j < 8; ++j) v[j] = (T)((float)v[j] + (float)r[j]);
                }
                *(V8*)(cbase + (long)row * ldc) = v;
            } else if (row < rows_left && cols_left >= 8) {
                // C's rows (and the residual's) may start at any element: the 16 bytes move as a copy of no stated
                // alignment, for which the compiler still issues one 16-byte access (global memory takes unaligned ones)
                if (R != nullptr) {
                    V8 r;
                    __builtin_memcpy(&r, rbase + (long)row * ldr, 16);
#pragma unroll
                    for (int j = 0; j < 8; ++j) v[j] = (T)((float)v[j] + (float)r[j]);
                }
                __builtin_memcpy(cbase + (long)row * ldc, &v, 16);
            } else if (row < rows_left) {
                // the last columns of a C whose width is not a multiple of 8: element by element
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (j < cols_left) {
                        T x = v[j];
                        if (R != nullptr) x = (T)((float)x + (float)rbase[(long)row * ldr + j]);
                        cbase[(long)row * ldc + j] = x;
                    }
            }
        }
    }
}

// Merges the partial tiles of a split-K launch without counters: C = sum over the ranges, in their order (+ R after the
// rounding, as in the epilogue). A thread takes 8 columns of a row. Bandwidth-bound: every partial tile is read once, mostly
// from the memory-side cache, by all CUs, where the last workgroup of a tile would read its tile's parts alone.
template <typename T>
static __global__ __launch_bounds__(256) void hgemm_merge_kernel(const float* __restrict__ part, T* C, const T* R, int M, int N, long mp, long np,
                                                          long ldc, long ldr, int splits) {
    using V8 = typename Elem<T>::v8;
    const int chunks = (int)(np / 8);
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    const long row = i / chunks;
    const int col = (int)(i - row * chunks) * 8;
    if (row >= M || col >= N) return;
    const float* p = part + row * np + col;
    float4v lo = *(const float4v*)p, hi = *(const float4v*)(p + 4);
    int r = 1;
    for (; r + 2 < splits; r += 3) {   // three ranges in flight
        float4v a[3], b[3];
#pragma unroll
        for (int u = 0; u < 3; ++u) {
            a[u] = *(const float4v*)(p + (r + u) * mp * np);
            b[u] = *(const float4v*)(p + (r + u) * mp * np + 4);
        }
#pragma unroll
        for (int u = 0; u < 3; ++u) { lo += a[u]; hi += b[u]; }
    }
    for (; r < splits; ++r) {
        lo += *(const float4v*)(p + r * mp * np);
        hi += *(const float4v*)(p + r * mp * np + 4);
    }
    V8 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[j] = (T)lo[j]; v[4 + j] = (T)hi[j]; }
    T* c = C + row * ldc + col;
    const T* res = R + row * ldr + col;
    if (col + 8 <= N) {
        if (R != nullptr) {
            V8 x;
            __builtin_memcpy(&x, res, 16);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = (T)((float)v[j] + (float)x[j]);
        }
        __builtin_memcpy(c, &v, 16);
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (col + j < N) c[j] = R != nullptr ? (T)((float)v[j] + (float)res[j]) : v[j];
    }
}

}  // namespace mi355
