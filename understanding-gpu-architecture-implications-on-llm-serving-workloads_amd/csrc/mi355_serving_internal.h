// Internal C++ entry points behind the C ABI of include/mi355_serving.h.
#pragma once
#include <hip/hip_runtime.h>
#include <atomic>
#include <cstddef>
#include <mutex>
#include "../../include/mi355_serving.h"

namespace mi355 {

// Raises a kernel's dynamic LDS limit once per device (the attribute belongs to the device the call is made on).
// Threads may race to set it; the call is idempotent, so the flags only need to be atomic.
struct DynamicLdsOnce {
    static constexpr int kMaxDevices = 64;
    std::atomic<bool> done[kMaxDevices] = {};
    hipError_t ensure(const void* kernel, int bytes) {
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        const bool tracked = dev >= 0 && dev < kMaxDevices;
        if (tracked && done[dev].load(std::memory_order_acquire)) return hipSuccess;
        e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e == hipSuccess && tracked) done[dev].store(true, std::memory_order_release);
        return e;
    }
};

// Launches the GEMM kernels; arguments as mi355_hgemm_add after validation (R == nullptr: no residual).
// `variant` pins a tile shape instead of the choice by shape (0); see mi355_internal_hgemm_variant below. `workspace`
// (16-byte aligned device memory, may be null): where aligned copies of operands with unaligned rows may be kept.
hipError_t hgemm_dispatch(const void* A, const void* B, void* C, const void* R, int M, int N, int K, long lda, long ldb,
                          long ldc, long ldr, int layout, int dtype, int variant, void* workspace, size_t workspace_bytes,
                          hipStream_t stream);

// The kernels of one element type and layout (hgemm.hip, one translation unit each).
template <typename T, int LAYOUT>
hipError_t gemm_layout(const void* A, const void* B, void* C, const void* R, int M, int N, int K, long lda, long ldb, long ldc,
                       long ldr, int variant, hipStream_t stream);
template <typename T, int LAYOUT>
hipError_t gemm_silu_mul_layout(const void* A, const void* B, void* C, int M, int N2, int K, long lda, long ldb, long ldc,
                                int variant, hipStream_t stream);

// The first two products of a layer's generation step (layout NT, few rows) with what stands around them.
struct RopeEpilogue {   // behind the QKV projection, as mi355_rope_qkv takes it
    void* kv_out;
    long o_batch, o_row, o_head;
    const float *cos_t, *sin_t;
    const int* positions;
    long pos_batch;
    int n_pos, S, q_heads, kv_heads;
};
struct NormPrologue {   // RMSNorm of the rows; weight == nullptr: none
    const void* weight;
    float eps;
};
template <typename T>
hipError_t gemm_step_qkv(const void* x, const NormPrologue& norm, const void* w, void* qkv, int M, int N, int K, long ldx, long ldb, long ldc,
                         const RopeEpilogue& rope, hipStream_t stream);
template <typename T>
hipError_t gemm_step_gate_up(const void* x, const NormPrologue& norm, const void* w, void* out, int M, int N, int K, long ldx, long ldb, long ldc,
                             hipStream_t stream);
hipError_t gemm_step_qkv_dispatch(const void* x, const NormPrologue& norm, const void* w, void* qkv, int M, int N, int K, const RopeEpilogue& rope,
                                  int dtype, hipStream_t stream);   // rows side by side
hipError_t gemm_step_gate_up_dispatch(const void* x, const NormPrologue& norm, const void* w, void* out, int M, int N, int K, int dtype,
                                      hipStream_t stream);

// The kernel of a product (hgemm_choice.hip); the shapes' numbers are those of mi355_internal_hgemm_variant below.
enum KernelShape { kTile256x256 = 1, kTile128x128, kTileHalf, kTile64x64, kTile128x256, kTile256x128, kTile32x64, kSmallM, kDeepRing, kDirect64x64, kDirect128x128 };
struct KernelChoice {
    int shape = kTile128x128;
    int splits = 1;           // ranges of K
    int wide_ranges = 0;      // kSmallM, layouts NN and TN: ranges of K of hgemm_smallm_wide_kernel, 0 = the kernel of 64 columns
    bool own_merge = false;   // their partial tiles are merged by a kernel of their own
    float us = 0.f;           // expected time
};
// a_kc, b_kc: the operand's K index is contiguous. tiles_ok, split_ok: the tiled kernels, ranges of K may be chosen. whole_lines: the
// second operand's rows are multiples of 128 bytes. gate_up: among the shapes whose waves hold 64 columns, the gate and the up
// of the same outputs. shape 0: none of these kernels.
KernelChoice choose_kernel(int M, int N, int K, bool a_kc, bool b_kc, bool tiles_ok, bool split_ok, bool whole_lines, bool gate_up = false);

// Row tiles per workgroup of the small-M kernel that keeps the activation rows in registers (hgemm_smallm_nt_rega_kernel), or 0 when
// it does not apply: K = 4096, at most 16 rows, whole tiles, and at
// least 192 workgroups left to keep the memory system busy. Measured on weights that come from HBM (a different weight
// matrix on every launch), against one tile per workgroup: 16 x 14336 x 4096 24.5 -> 21.7 us with four tiles (22.1 with
// two), 16 x 6144 x 4096 13.1 -> 11.4 (two), 16 x 28672 x 4096 43.2 -> 40.5 (four; 42.2 with two). Up to 8 rows, where
// the activation slab is half as large to begin with: 8 x 14336 x 4096 22.3 -> 20.5 us with two tiles (21.2 with four),
// 8 x 28672 x 4096 39.1 -> 39.4-39.9 either way, so the widest products keep one tile per workgroup there.
inline int smallm_nt_rega_tpw(int M, int n_tiles, int K, long lda, long ldb) {
    if (M > 16 || K != 4096 || lda >= (1L << 22) || ldb >= (1L << 22)) return 0;   // lane offsets of up to 72 rows in 32 bits
    if (M <= 8) return n_tiles % 2 == 0 && n_tiles / 2 >= 192 && n_tiles / 2 <= 512 ? 2 : 0;
    for (int tpw : {4, 2})
        if (n_tiles % tpw == 0 && n_tiles / tpw >= 192) return tpw;
    return 0;
}

// Device memory for a workspace of the library; another stream's capture does not notice.
hipError_t workspace_malloc(void** out, size_t bytes);
// Workspace of the split-K path: ticket counters (one per tile, at zero between launches), then `bytes` minus those for
// partial tiles. hipErrorStreamCaptureUnsupported / hipErrorOutOfMemory: none to be had.
constexpr size_t kSplitKCounterBytes = 16 * 1024;   // up to 4096 tiles
hipError_t split_k_workspace(size_t bytes, hipStream_t stream, char** out, std::unique_lock<std::mutex>* order);
#ifdef MI355_TIMELINE
extern hipError_t (*timeline_hgemm_reader)(void*, size_t);   // of the translation unit whose tiled kernel was launched last
#endif

// Aligned copies of GEMM operands (gemm_pack.hip): which operands need one, and the rows and bytes of the copies.
struct GemmPackPlan {
    struct Operand {
        bool pack = false;
        int cols = 0;       // elements of a stored row
        long ld = 0;        // row stride of the copy (of the operand itself where none is made)
        size_t bytes = 0;   // of the copy
    };
    Operand a, b;
    size_t b_offset() const { return (a.bytes + 255) / 256 * 256; }   // where B's copy starts behind A's
    size_t bytes() const { return b_offset() + b.bytes; }
};
GemmPackPlan gemm_pack_plan(const void* A, const void* B, int M, int N, int K, long lda, long ldb, int layout);
hipError_t gemm_pack_launch(const GemmPackPlan& plan, const void* A, const void* B, long lda, long ldb, void* a_copy, void* b_copy,
                            hipStream_t stream);
// The product of operands of any alignment and stride (hgemm_direct.hip): by shape (variant 0), or a pinned kernel. And the tiles and
// ranges of K that it takes by shape.
KernelChoice choose_direct(int M, int N, int K, int layout, bool split_ok);
hipError_t gemm_direct_dispatch(const void* A, const void* B, void* C, const void* R, int M, int N, int K, long lda, long ldb, long ldc, long ldr,
                                int layout, int dtype, int variant, hipStream_t stream);
// Bytes of workspace the public query asks for (0: none, nothing to copy or not worth it), and those that the copies of a call take.
size_t hgemm_workspace_bytes(const void* A, const void* B, int M, int N, int K, long lda, long ldb, int layout);
size_t hgemm_copy_bytes(const void* A, const void* B, int M, int N, int K, long lda, long ldb, int layout);

// Element strides of the attention operands: tensor[b][h][s][d] lives at b*batch + h*head + s*row + d (d contiguous).
struct FmhaStrides {
    long q_batch, q_head, q_row;
    long k_batch, k_head, k_row;
    long v_batch, v_head, v_row;
    long o_batch, o_head, o_row;
};

// The product fused with silu(gate) * up (see hgemm_main_kernel's EPI); hipErrorNotSupported for shapes without it.
hipError_t hgemm_silu_mul_dispatch(const void* A, const void* B, void* C, int M, int N2, int K, long lda, long ldb, long ldc,
                                   int layout, int dtype, int variant, hipStream_t stream);

// Where the split-KV and key-range attention paths keep their partial results.
struct FmhaWorkspace {
    enum Kind { kLibrary, kCaller, kStatic };
    Kind kind = kLibrary;     // kLibrary: the library's own grow-only buffer of (device, stream)
    void* ptr = nullptr;      // kCaller: device memory of the caller, `bytes` long
    size_t bytes = 0;         // kStatic: the fixed-size __device__ array of fmha_decode.hip (nothing is ever allocated)
};

// Launches the attention forward kernels; arguments as mi355_fmha_fwd_strided after validation.
// `variant` pins a kernel instead of the choice by shape (0); see mi355_internal_fmha_fwd_variant below.
hipError_t fmha_fwd_dispatch(const void* Q, const void* K, const void* V, void* O, float* LSE, int B, int Hq, int Hkv,
                             int Sq, int Sk, float scale, int causal, int kv_valid_len, const FmhaStrides& strides,
                             int dtype, int variant, const FmhaWorkspace& ws, hipStream_t stream);

// Split-KV path for few query rows per kv head (generation step); see fmha_decode.hip.
bool fmha_decode_applicable(int B, int Hq, int Hkv, int Sq, int Sk, int kv_valid_len);
// Key ranges per (batch, kv head), 0 where a call does not take that path, and waves per workgroup.
void fmha_decode_plan_of(int B, int Hq, int Hkv, int Sq, int kv_valid_len, int* splits, int* waves);
// Bytes of workspace a caller is asked for (0 when a call with these sizes does not take the split-KV path, or has one range).
size_t fmha_decode_workspace_bytes(int B, int Hq, int Hkv, int Sq, int Sk, int kv_valid_len);
// Bytes of workspace the key-range path of fmha_fwd.hip uses for a call with these sizes (0 when it does not take it), and
// the bytes a call uses on whichever of the two paths it takes.
size_t fmha_key_range_workspace_bytes(int B, int Hq, int Hkv, int Sq, int Sk, int kv_valid_len);
size_t fmha_workspace_bytes(int B, int Hq, int Hkv, int Sq, int Sk, int kv_valid_len);
// Size of the static scratch array behind FmhaWorkspace::kStatic.
size_t fmha_decode_static_scratch_bytes();
template <typename T>
hipError_t fmha_decode_dispatch(const T* Q, const T* K, const T* V, T* O, float* LSE, int B, int Hq, int Hkv, int Sq, int Sk,
                                float scale, int causal, int kv_valid_len, const FmhaStrides& strides, const FmhaWorkspace& ws,
                                hipStream_t stream);

// Layer glue (glue.hip); arguments as the mi355_rmsnorm / mi355_rope / mi355_silu_mul entry points after validation.
hipError_t rmsnorm_dispatch(const void* x, const void* residual, void* res_out, const void* weight, void* out, long rows,
                            int hidden, long ldx, long ldr, long ldro, long ldo, float eps, int dtype, hipStream_t stream);
// rope_dispatch: `heads` heads are rotated, the first `inplace_heads` of them in place, `copy_heads` more are copied;
// consecutive heads of `out` lie o_head elements apart.
hipError_t rope_dispatch(const void* x, void* out, int B, int S, int inplace_heads, int heads, int copy_heads, long x_batch,
                         long x_row, long o_batch, long o_row, long o_head, const float* cos_t, const float* sin_t, const int* positions, long pos_batch,
                         int n_pos, int dtype, hipStream_t stream);
hipError_t silu_mul_dispatch(const void* in, void* out, long rows, int inter, int block, long ld_in, long ld_out, int dtype,
                             hipStream_t stream);

}  // namespace mi355

// Test and tuning hooks: exported from the shared library but not part of its public header. They take the kernel
// variant as an argument (no process-wide state). Where a layout lacks a pinned kernel, or the operands' rows are not aligned, the
// choice by shape takes its place; of more ranges than K has tiles as many are taken as it has.
//   gemm: 0 = by shape; 1 = 256x256 tiles, 2 = 128x128, 3 = 64x128 (layout NT: 128x64), 4 = 64x64 with a ring of four
//         stages, 5 = 128x256, 6 = 256x128, 7 = 32x64 (layouts NN and NT), 8 = the small-M kernels (up to 64 rows), 9 = 64x64 with
//         a ring of eight; shapes 1 .. 7 take s ranges of K with variant + 16 s, merged by a kernel of their own (instead of
//         the last workgroup of a tile) with variant + 16 s + 4096, shape 1 always; 8 + 16 s (layouts NN and TN, s > 1) = 128 columns and
//         s ranges of K, merged by the last workgroup of a tile. 10, 11 = the direct kernel for operands of any
//         alignment on 64x64 and 128x128 tiles, s ranges of K with + 16 s. The gate/up product: 1, 2, 4, 5, 6, 8, 9
//   fmha: 0 = by shape, 1 = 128-query workgroups, 2 = 256-query workgroups (1 and 2 also keep generation-step shapes off
//         the split-KV path), 3 = keys of a long cache cut into ranges and merged, 4 = those of a shorter one, partial results in 32 bits
//         (an error where the choice by shape would not do that)
extern "C" {
int mi355_internal_hgemm_variant(const void* A, const void* B, void* C, int M, int N, int K, int64_t lda, int64_t ldb,
                                 int64_t ldc, int layout, int dtype, int variant, void* stream);
// with a residual R (arguments as mi355_hgemm_add)
int mi355_internal_hgemm_add_variant(const void* A, const void* B, const void* R, void* C, int M, int N, int K, int64_t lda, int64_t ldb,
                                     int64_t ldr, int64_t ldc, int layout, int dtype, int variant, void* stream);
// the variant that the choice by shape takes for a product of 16-byte aligned operands (ldb: row stride of the second one), and the
// time it expects (us may be null); for the small-M kernels (8) in layouts NN and TN the second says which: ranges of K of the 128-column
// kernel, to be pinned with 8 + 16 ranges, or 0, the 64-column kernel
int mi355_internal_hgemm_choice(int M, int N, int K, int64_t ldb, int layout, float* us);
int mi355_internal_hgemm_wide_ranges(int M, int N, int K, int64_t ldb, int layout);
int mi355_internal_hgemm_silu_mul_variant(const void* A, const void* B, void* C, int M, int N, int K, int64_t lda, int64_t ldb,
                                          int64_t ldc, int layout, int dtype, int variant, void* stream);
int mi355_internal_fmha_fwd_variant(const void* Q, const void* K, const void* V, void* O, float* LSE, int B, int Hq, int Hkv,
                                    int Sq, int Sk, int D, float scale, int causal, int kv_valid_len, const int64_t* strides,
                                    int dtype, int variant, void* stream);
// the variant of the direct kernel that a product of unaligned operands takes if it is not copied, and the time it expects (us may be null)
int mi355_internal_hgemm_direct_choice(int M, int N, int K, int layout, float* us);
// bytes of workspace that mi355_gemm_ws uses for a call (0: it makes no copies): what the operators, the Python binding and the decoder layer
// allocate, where mi355_gemm_workspace_bytes may ask for more
size_t mi355_internal_gemm_copy_bytes(const void* A, const void* B, int M, int N, int K, int64_t lda, int64_t ldb, int layout);
// The QKV projection of a generation step's layer with the RMSNorm of its rows (norm_weight null: none) and mi355_rope_qkv in one
// launch: qkv = rope(rmsnorm(x) w_qkv^T), rotated keys and values into kv_out; x is [B, S, hidden], qkv [B, S, (q_heads + 2 kv_heads)
// * 128]. And silu(gate) * up of the normalised rows (w_gu in groups of 32 gate and 32 up rows). The bits of the single launches on
// the small-M kernel. MI355_ERR_UNSUPPORTED (no error text): nothing was launched, take the single calls.
int mi355_internal_step_qkv(const void* x, const void* norm_weight, float eps, const void* w_qkv, void* qkv, void* kv_out, int B, int S, int q_heads,
                            int kv_heads, int hidden, int64_t out_batch, int64_t out_row, int64_t out_head, const float* cos_table,
                            const float* sin_table, const int32_t* positions, int64_t pos_batch, int n_positions, int dtype, void* stream);
int mi355_internal_step_gate_up(const void* x, const void* norm_weight, float eps, const void* w_gu, void* out, int rows, int inter, int hidden,
                                int dtype, void* stream);
// how few queries over `kv_valid_len` keys are cut: key ranges per (batch, kv head), 0 = by the prefill kernel; waves per workgroup
int mi355_internal_fmha_decode_plan(int B, int Hq, int Hkv, int Sq, int kv_valid_len, int* splits, int* waves);
}
