// GEMM over operands of any alignment and stride, read where they lie.
//
// The tiled kernels of hgemm.hip move 16 aligned bytes straight into LDS. An operand whose rows are not 16-byte aligned (a dense
// matrix whose row length is not a multiple of 8, a view that starts at an odd element) would need an aligned copy first
// (gemm_pack.hip): a launch, and the operand written and read once more. Here it goes through registers instead:
//   * a thread reads 16 bytes at any element (global memory takes such loads) and stores them to LDS in the tiled kernels' layout,
//     kDepth K tiles ahead, so a load has that many K tiles to come back in; the LDS tiles are double buffered, one barrier per K tile;
//   * no load has a condition: an offset past the last whole 16 bytes of the operand is moved back to it, and what that changes
//     (only chunks of the last two K tiles that count) is put right on the way to LDS: elements moved down, zeros behind K;
//   * fragments, products and the stores of C are those of the tiled kernels, four waves side by side over the tile. What bounds it is
//     the CU's vector memory path, which takes 53 cycles for a load of 64 unaligned 16-byte pieces: it is busy 94 % of a CU's cycles on
//     64x64 tiles (.41 us a K tile) and 73 .. 88 % on 128x128 (.83), LDS 29 and 25 %, the matrix pipes 14 and 24 % (1999 x 3001 x 2503 NN).
//     Rows 2 bytes off a multiple of 4 take 20 - 25 % longer than aligned ones.
// us per product, aligned copies in front of the tiled kernels / direct: 1 x 203 x 236 TN 8.1 / 5.3, 8 x 6407 x 983 NN 19.2 / 10.5, 397 x 965 x 313
// NN 10.9 / 6.8, 99 x 9001 x 3021 NT 43 / 30, 62 x 19578 x 5867 NT 168 / 78; large ones stay with the copies (1999 x 3001 x 2503 NN 43 / 59).
// Operands of fewer than 8 elements are read one element at a time.
#include <algorithm>
#include <mutex>
#include "hgemm_tiles.h"
#include "mi355_common.h"
#include "mi355_serving_internal.h"

namespace mi355 {
namespace {

constexpr int kDirectThreads = 256;
constexpr int kDirectWaves = 4;

// the 8 elements of a chunk moved `by` elements down, zeros from above (by >= 8: all zeros)
__device__ __forceinline__ int4v moved_down(int4v v, int by) {
    const uint64_t lo = (uint64_t)(uint32_t)v[0] | (uint64_t)(uint32_t)v[1] << 32, hi = (uint64_t)(uint32_t)v[2] | (uint64_t)(uint32_t)v[3] << 32;
    const int bits = 16 * by;
    const uint64_t l = by == 0 ? lo : by < 4 ? (lo >> bits) | (hi << (64 - bits)) : by < 8 ? hi >> (bits - 64) : 0;
    const uint64_t h = by < 4 ? hi >> bits : 0;
    return int4v{(int)(uint32_t)l, (int)(uint32_t)(l >> 32), (int)(uint32_t)h, (int)(uint32_t)(h >> 32)};
}

// One operand's share of a thread: kChunks 16-byte chunks of every K tile. KC: its K index is contiguous. ROWS: rows of the
// product (columns of it for the second operand) in a tile. SINGLE: the operand may have fewer than 8 elements.
template <typename T, bool KC, int ROWS, int DEPTH, bool SINGLE>
struct DirectOperand {
    using Kc = KContigTile<ROWS, 64, kDirectWaves>;
    using Mn = MNContigTile<ROWS, 64, kDirectWaves>;
    static constexpr int kPerRow = KC ? 8 : ROWS / 8;                 // chunks of a stored row
    static constexpr int kStep = kDirectThreads / kPerRow;            // stored rows between a thread's chunks
    static constexpr int kChunks = ROWS * 64 / 8 / kDirectThreads;
    static constexpr int kBytes = ROWS * 64 * 2;
    const T* base;
    long last;            // offset of the operand's last 8 elements; negative: fewer than 8 elements
    long first, apart, ahead;   // element offset of the thread's first chunk in K tile 0, between its chunks, per K tile
    int k_first;          // k of the first chunk
    int lds;              // byte offset of the first chunk in the LDS tile (the others lie kStep rows on: the swizzle repeats)
    int4v v[DEPTH][kChunks];

    __device__ __forceinline__ DirectOperand(const T* p, long ld, long row0, int rows, int K, int tid) {
        const int r = tid / kPerRow, c = tid % kPerRow;
        base = p;
        last = KC ? (rows - 1) * ld + K - 8 : (K - 1) * ld + rows - 8;
        first = KC ? (row0 + r) * ld + c * 8 : r * ld + row0 + c * 8;
        apart = kStep * ld;
        ahead = KC ? 64 : 64 * ld;
        k_first = KC ? c * 8 : r;
        if constexpr (KC) lds = r * Kc::kRowBytes + ((c ^ Kc::swz(r)) << 4);
        else lds = r * Mn::kRowBytes + ((c ^ Mn::swz(r)) << 4);
        static_assert(kStep % 16 == 0, "rows kStep apart have the same swizzle");
    }
    template <int STAGE>
    __device__ __forceinline__ void load(int kt) {
#pragma unroll
        for (int i = 0; i < kChunks; ++i) {
            const long off = first + i * apart + kt * ahead;
            if constexpr (SINGLE) v[STAGE][i] = single_elements(off);
            else __builtin_memcpy(&v[STAGE][i], base + min(off, last), 16);
        }
    }
    // END: maybe one of the last two K tiles of the product; `left` elements of K exist from the tile's first on
    template <int STAGE, bool END>
    __device__ __forceinline__ void store(MI355_LDS char* tile, int kt, int left) {
#pragma unroll
        for (int i = 0; i < kChunks; ++i) {
            int4v x = v[STAGE][i];
            if constexpr (END) {
                if constexpr (!SINGLE) x = moved_down(x, (int)min(8L, max(0L, first + i * apart + kt * ahead - last)));
                if constexpr (KC) x = __builtin_bit_cast(int4v, first_of_chunk(__builtin_bit_cast(half8, x), left - k_first));
                else if (k_first + i * kStep >= left) x = int4v{0, 0, 0, 0};
            }
            *(MI355_LDS int4v*)(tile + lds + i * kStep * (KC ? Kc::kRowBytes : Mn::kRowBytes)) = x;
        }
    }
    __device__ __forceinline__ int4v single_elements(long off) const {
        const uint16_t* const e = reinterpret_cast<const uint16_t*>(base);
        uint64_t lo = 0, hi = 0;
#pragma unroll 1
        for (int j = 0; j < 8 && off + j < last + 8; ++j) {
            const uint64_t x = e[off + j];
            if (j < 4) lo |= x << (16 * j);
            else hi |= x << (16 * (j - 4));
        }
        return int4v{(int)(uint32_t)lo, (int)(uint32_t)(lo >> 32), (int)(uint32_t)hi, (int)(uint32_t)(hi >> 32)};
    }
    // the fragment of 16 rows from row0 on, k = 32 kk .. + 31
    static __device__ __forceinline__ half8 fragment(MI355_LDS const char* tile, int row0, int kk, int lane) {
        if constexpr (KC) {
            return lds_read_b128(tile + Kc::frag_offset(row0, kk, lane));
        } else {
            MI355_LDS const char* const p = tile + Mn::frag_offset(row0, lane) + kk * 32 * Mn::kRowBytes;
            return concat(lds_read_tr16_b64(p), lds_read_tr16_b64(p + 4 * Mn::kRowBytes));
        }
    }
};

// part: null, or where the partial tiles of ranges of K go, rows of a padded matrix per range (merged by hgemm_merge_kernel)
template <typename T, bool A_KC, bool B_KC, int TILE, int DEPTH, bool SINGLE>
__global__ __launch_bounds__(kDirectThreads) void hgemm_direct_kernel(const T* __restrict__ A, const T* __restrict__ B, T* C, const T* R, int M, int N,
                                                                      int K, long lda, long ldb, long ldc, long ldr, float* part) {
    using OpA = DirectOperand<T, A_KC, TILE, DEPTH, SINGLE>;
    using OpB = DirectOperand<T, B_KC, TILE, DEPTH, SINGLE>;
    constexpr int kBlocks = TILE / 32;   // a wave's sub-tile: kBlocks x kBlocks blocks of 16x16
    constexpr int kBuffer = OpA::kBytes + OpB::kBytes;
    __shared__ __attribute__((aligned(16))) char smem_[2 * kBuffer];
    MI355_LDS char* const smem = (MI355_LDS char*)smem_;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    // an XCD takes neighbouring tiles, rows of tiles first, so that the tiles of a column of them find their B in its L2
    const int tiles_m = (M + TILE - 1) / TILE, tiles = tiles_m * ((N + TILE - 1) / TILE);
    const int tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int tile_n = tile / tiles_m, tile_m = tile - tile_n * tiles_m;
    const long m0 = (long)tile_m * TILE, n0 = (long)tile_n * TILE;
    const int ktiles = (K + 63) / 64, per_range = (ktiles + gridDim.y - 1) / gridDim.y;
    const int kt_begin = blockIdx.y * per_range, kt_end = min(kt_begin + per_range, ktiles);

    OpA a(A, lda, m0, M, K, tid);
    OpB b(B, ldb, n0, N, K, tid);
    float4v acc[kBlocks][kBlocks];
#pragma unroll
    for (int i = 0; i < kBlocks; ++i)
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};

    static_for<0, DEPTH>([&](auto d) {
        const int kt = min(kt_begin + (int)d, ktiles - 1);
        a.template load<d>(kt);
        b.template load<d>(kt);
    });
    const auto step = [&](auto d, auto maybe_end, int kt) __attribute__((always_inline)) {
        MI355_LDS char* const sa = smem + (kt & 1) * kBuffer;
        MI355_LDS char* const sb = sa + OpA::kBytes;
        a.template store<d, maybe_end>(sa, kt, K - kt * 64);
        b.template store<d, maybe_end>(sb, kt, K - kt * 64);
        const int next = min(kt + DEPTH, kt_end - 1);
        a.template load<d>(next);
        b.template load<d>(next);
        // every wave's part of this tile is in LDS, and no wave reads the other buffer any more
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            typename Elem<T>::v8 af[kBlocks], bf[kBlocks];
#pragma unroll
            for (int i = 0; i < kBlocks; ++i) af[i] = Elem<T>::frag(OpA::fragment(sa, (wm * kBlocks + i) * 16, kk, lane));
#pragma unroll
            for (int j = 0; j < kBlocks; ++j) bf[j] = Elem<T>::frag(OpB::fragment(sb, (wn * kBlocks + j) * 16, kk, lane));
#pragma unroll
            for (int i = 0; i < kBlocks; ++i)
#pragma unroll
                for (int j = 0; j < kBlocks; ++j) acc[i][j] = Elem<T>::mfma16(bf[j], af[i], acc[i][j]);
        }
    };
    int kt = kt_begin;
    for (const int whole = min(kt_end, ktiles - 2); kt + DEPTH <= whole; kt += DEPTH)
        static_for<0, DEPTH>([&](auto d) __attribute__((always_inline)) { step(d, std::false_type{}, kt + (int)d); });
    static_for<0, DEPTH + 1>([&](auto d) __attribute__((always_inline)) {
        if (kt + (int)d < kt_end) step(std::integral_constant<int, d % DEPTH>{}, std::true_type{}, kt + (int)d);
    });

    const long row0 = m0 + wm * kBlocks * 16, col0 = n0 + wn * kBlocks * 16;
    if (part != nullptr) {
        const long mp = (long)tiles_m * TILE, np = (long)(tiles / tiles_m) * TILE;
        float* const dst = part + (blockIdx.y * mp + row0 + (lane & 15)) * np + col0 + 4 * (lane >> 4);
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
#pragma unroll
            for (int j = 0; j < kBlocks; ++j) *(float4v*)(dst + i * 16 * np + j * 16) = acc[i][j];
        return;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // the tiles have been read: their memory holds the sub-tiles of C now
    store_wave_tile<T, kBlocks, kBlocks, 0, true>(acc, smem + wave * (kBlocks * kBlocks * 512), C, R, row0, col0, M, N, ldc, ldr, lane);
}

template <typename T, bool A_KC, bool B_KC, int TILE, int DEPTH, bool SINGLE = false>
hipError_t launch_direct(const T* A, const T* B, T* C, const T* R, int M, int N, int K, long lda, long ldb, long ldc, long ldr, int splits,
                         hipStream_t stream) {
    const long tiles_m = (M + TILE - 1) / TILE, tiles_n = (N + TILE - 1) / TILE, tiles = tiles_m * tiles_n;
    const dim3 grid((unsigned)((tiles + 7) / 8 * 8), (unsigned)splits);
    if (splits <= 1) {
        hgemm_direct_kernel<T, A_KC, B_KC, TILE, DEPTH, SINGLE><<<grid, dim3(kDirectThreads), 0, stream>>>(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, nullptr);
        return hipGetLastError();
    }
    char* ws = nullptr;
    std::unique_lock<std::mutex> order;   // the launches below follow one another on the stream
    const size_t bytes = kSplitKCounterBytes + (size_t)tiles * splits * TILE * TILE * 4;
    if (hipError_t e = split_k_workspace(bytes, stream, &ws, &order); e != hipSuccess) return e;
    float* const part = reinterpret_cast<float*>(ws + kSplitKCounterBytes);
    hgemm_direct_kernel<T, A_KC, B_KC, TILE, DEPTH, SINGLE><<<grid, dim3(kDirectThreads), 0, stream>>>(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, part);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    const long np = tiles_n * TILE, chunks = (long)M * (np / 8);
    hgemm_merge_kernel<T><<<dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, stream>>>(part, C, R, M, N, tiles_m * TILE, np, ldc, ldr, splits);
    return hipGetLastError();
}

template <typename T>
hipError_t direct_of_type(const void* A, const void* B, void* C, const void* R, int M, int N, int K, long lda, long ldb, long ldc, long ldr,
                          int layout, int shape, int splits, hipStream_t stream) {
    const auto go = [&](auto a_kc, auto b_kc) {
        const long span_a = a_kc ? (M - 1) * lda + K : (K - 1) * lda + M, span_b = b_kc ? (N - 1) * ldb + K : (K - 1) * ldb + N;
        const auto launch = std::min(span_a, span_b) < 8 ? &launch_direct<T, a_kc, b_kc, 64, 1, true>
                            : shape == kDirect128x128    ? &launch_direct<T, a_kc, b_kc, 128, 2>
                                                         : &launch_direct<T, a_kc, b_kc, 64, 4>;
        return launch(static_cast<const T*>(A), static_cast<const T*>(B), static_cast<T*>(C), static_cast<const T*>(R), M, N, K, lda, ldb, ldc, ldr,
                      splits, stream);
    };
    if (layout == MI355_GEMM_TN) return go(std::false_type{}, std::false_type{});
    return layout == MI355_GEMM_NT ? go(std::true_type{}, std::true_type{}) : go(std::true_type{}, std::false_type{});
}

}  // namespace

hipError_t gemm_direct_dispatch(const void* A, const void* B, void* C, const void* R, int M, int N, int K, long lda, long ldb, long ldc, long ldr,
                                int layout, int dtype, int variant, hipStream_t stream) {
    if (layout != MI355_GEMM_NN && layout != MI355_GEMM_NT && layout != MI355_GEMM_TN) return hipErrorInvalidValue;
    const auto run = [&](int shape, int splits) {
        const int ktiles = (K + 63) / 64, per_range = (ktiles + splits - 1) / splits;
        const auto entry = dtype == MI355_DTYPE_BF16 ? &direct_of_type<bf16_t> : &direct_of_type<half_t>;
        return entry(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, layout, shape, (ktiles + per_range - 1) / per_range, stream);   // each range holds a K tile
    };
    if (variant != 0) return run(variant & 15, std::max(1, variant >> 4 & 0xff));
    KernelChoice pick = choose_direct(M, N, K, layout, true);
    const hipError_t e = run(pick.shape, pick.splits);
    if (pick.splits <= 1 || (e != hipErrorStreamCaptureUnsupported && e != hipErrorOutOfMemory)) return e;
    (void)hipGetLastError();   // no workspace to be had: the whole of K in every workgroup
    pick = choose_direct(M, N, K, layout, false);
    return run(pick.shape, 1);
}

}  // namespace mi355
