// Host side of the GEMM entry points: aligned copies of operands, the choice of the translation unit that holds the kernels
// of an element type and layout (hgemm.hip), and the workspace of the split-K path.
#include <cmath>
#include <map>
#include <mutex>
#include <utility>
#include "mi355_common.h"
#include "mi355_serving_internal.h"

namespace mi355 {

static __global__ void hgemm_clear_kernel(unsigned* p, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0u;
}

// hipMalloc in relaxed capture mode: in the thread's own (global) mode an allocation while any other stream is being captured fails and
// invalidates that capture, and a first call on one stream would end what another one records.
hipError_t workspace_malloc(void** out, size_t bytes) {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    if (hipError_t e = hipThreadExchangeStreamCaptureMode(&mode); e != hipSuccess) return e;
    const hipError_t e = hipMalloc(out, bytes);
    const hipError_t back = hipThreadExchangeStreamCaptureMode(&mode);
    return e != hipSuccess ? e : back;
}

// The workspace of the split-K path: one buffer per (device, stream), allocated at first use and replaced by a larger one when
// a call needs more; a buffer that has been handed to a kernel is never freed (a HIP graph captured earlier may hold its
// address). Nothing can be allocated while the stream is capturing: such a call (no buffer yet, or too small a one) fails
// with hipErrorStreamCaptureUnsupported and its caller takes the kernels without split-K instead. The ticket counters, in
// front of the partial tiles, are zeroed when a buffer is new (a fill kernel on the calling stream) and left at zero by
// every launch. `order` comes back holding the lock of that (device, stream): the caller keeps it until its launches are
// issued, so that of two threads with one stream neither's partial tiles are overwritten in front of the other's merge.
hipError_t split_k_workspace(size_t bytes, hipStream_t stream, char** out, std::unique_lock<std::mutex>* order) {
    struct Buf {
        void* ptr = nullptr;
        size_t size = 0;
        std::mutex order;
    };
    static std::mutex mu;
    static std::map<std::pair<int, hipStream_t>, Buf> bufs;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    Buf* entry = nullptr;
    {
        std::lock_guard<std::mutex> lock(mu);
        entry = &bufs[std::make_pair(dev, stream)];   // entries stay where they are
    }
    Buf& b = *entry;
    *order = std::unique_lock<std::mutex>(b.order);
    if (b.size < bytes) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        e = hipStreamIsCapturing(stream, &cap);
        if (e != hipSuccess) return e;
        if (cap != hipStreamCaptureStatusNone) return hipErrorStreamCaptureUnsupported;
        const size_t want = bytes < (size_t(8) << 20) ? (size_t(8) << 20) : bytes + bytes / 2;
        void* fresh_buf = nullptr;
        e = workspace_malloc(&fresh_buf, want);
        if (e != hipSuccess) return e;
        b.ptr = fresh_buf;   // the previous buffer, if any, stays allocated (see above)
        b.size = want;
        hgemm_clear_kernel<<<dim3(4), dim3(256), 0, stream>>>(static_cast<unsigned*>(b.ptr), (int)(kSplitKCounterBytes / sizeof(unsigned)));
        e = hipGetLastError();
        if (e != hipSuccess) {
            b.size = 0;   // counters not cleared: the next call starts over
            return e;
        }
    }
    *out = static_cast<char*>(b.ptr);
    return hipSuccess;
}

// Whether the copies of a plan are repaid: a launch, each copied operand read and written once, and the product on the kernels for
// aligned rows, against the direct kernel, which reads the operands where they lie. A product behind its copies, whose rows are no whole
// lines, takes longer than choose_kernel expects, by up to half of a short one: the terms fitted to 185 products with copies, both operands from
// HBM, rms 10 %. us, copies / direct: 2169 x 2399 x 1727 NT 34.5 / 47.7, 475 x 7131 x 4859 TN 64 / 77, 1999 x 3001 x 2503 NN 43 / 59, 751 x 385 x 8595
// NN 32 / 43; 99 x 9001 x 3021 NT 43 / 30, 8 x 6407 x 983 NN 19.2 / 10.5, 683 x 615 x 2587 NN 23.2 / 16.0, 62 x 19578 x 5867 NT 168 / 78. What the choice
// between them takes: choose_direct.
static bool copies_pay(const GemmPackPlan& plan, int M, int N, int K, int layout) {
    const KernelChoice fast = choose_kernel(M, N, K, layout != MI355_GEMM_TN, layout == MI355_GEMM_NT, true, true, plan.b.ld % 64 == 0);
    const float copied_mb = 2e-6f * (float)(plan.a.bytes + plan.b.bytes);
    const float copies_us = 3.8f + fast.us + (fast.splits > 1 ? .47f : .755f) * fminf(fast.us, 12.f) + copied_mb / 7.67f;
    return copies_us < choose_direct(M, N, K, layout, true).us;
}

size_t hgemm_copy_bytes(const void* A, const void* B, int M, int N, int K, long lda, long ldb, int layout) {
    if (K <= 64) return 0;
    const GemmPackPlan plan = gemm_pack_plan(A, B, M, N, K, lda, ldb, layout);
    if (!plan.a.pack && !plan.b.pack) return 0;
    return copies_pay(plan, M, N, K, layout) ? plan.bytes() : 0;
}

// The public query answers as it did when a workgroup per 64 x 64 outputs that gathers its operands 16 columns of K at a time (.0533 us per
// column of K, more where such workgroups wait for each other) was what such products ran on without copies: never less than the copies
// of the call take, and often more, as the direct kernel needs none for most of these products (hgemm_copy_bytes: 0 where this asks for
// 412 MB, 8 x 50257 x 4096 NN).
size_t hgemm_workspace_bytes(const void* A, const void* B, int M, int N, int K, long lda, long ldb, int layout) {
    if (K <= 64) return 0;
    const GemmPackPlan plan = gemm_pack_plan(A, B, M, N, K, lda, ldb, layout);
    if (!plan.a.pack && !plan.b.pack) return 0;
    if (plan.bytes() <= (size_t(1) << 20) || copies_pay(plan, M, N, K, layout)) return plan.bytes();
    const float wgs = (float)((M + 63) / 64) * (float)((N + 63) / 64), rows = (float)(M < 64 ? M : 64);
    const float per_wg = layout == MI355_GEMM_NT ? 1.94e-4f * (1.f + .0144f * rows) : 4.04e-5f * (1.f + (layout == MI355_GEMM_TN ? .0103f : .0559f) * rows);
    const float gather_us = 2.32f + (float)K * fmaxf(.0533f, per_wg * wgs);
    const KernelChoice fast = choose_kernel(M, N, K, layout != MI355_GEMM_TN, layout == MI355_GEMM_NT, true, true, plan.b.ld % 64 == 0);
    return fast.us + 5.3f + 2.f * (float)(plan.a.bytes + plan.b.bytes) / 5.96e6f < gather_us ? plan.bytes() : 0;
}

template <typename T>
static hipError_t gemm_of_type(const void* A, const void* B, void* C, const void* R, int M, int N, int K, long lda, long ldb, long ldc,
                               long ldr, int layout, int variant, hipStream_t stream) {
    switch (layout) {
        case MI355_GEMM_NN: return gemm_layout<T, MI355_GEMM_NN>(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, variant, stream);
        case MI355_GEMM_NT: return gemm_layout<T, MI355_GEMM_NT>(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, variant, stream);
        case MI355_GEMM_TN: return gemm_layout<T, MI355_GEMM_TN>(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, variant, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t hgemm_dispatch(const void* A, const void* B, void* C, const void* R, int M, int N, int K, long lda, long ldb,
                          long ldc, long ldr, int layout, int dtype, int variant, void* workspace, size_t workspace_bytes,
                          hipStream_t stream) {
    if ((variant & 15) == kDirect64x64 || (variant & 15) == kDirect128x128)
        return gemm_direct_dispatch(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, layout, dtype, variant, stream);
    if (const size_t need = workspace ? hgemm_copy_bytes(A, B, M, N, K, lda, ldb, layout) : 0; need > 0 && need <= workspace_bytes) {
        const GemmPackPlan plan = gemm_pack_plan(A, B, M, N, K, lda, ldb, layout);
        char* a_copy = static_cast<char*>(workspace);
        char* b_copy = a_copy + plan.b_offset();
        if (hipError_t e = gemm_pack_launch(plan, A, B, lda, ldb, a_copy, b_copy, stream); e != hipSuccess) return e;
        if (plan.a.pack) A = a_copy;
        if (plan.b.pack) B = b_copy;
        lda = plan.a.ld;
        ldb = plan.b.ld;
    }
    if (dtype == MI355_DTYPE_BF16) return gemm_of_type<bf16_t>(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, layout, variant, stream);
    return gemm_of_type<half_t>(A, B, C, R, M, N, K, lda, ldb, ldc, ldr, layout, variant, stream);
}

hipError_t hgemm_silu_mul_dispatch(const void* A, const void* B, void* C, int M, int N2, int K, long lda, long ldb, long ldc,
                                   int layout, int dtype, int variant, hipStream_t stream) {
    const bool bf16 = dtype == MI355_DTYPE_BF16, nn = layout == MI355_GEMM_NN;
    if (!nn && layout != MI355_GEMM_NT) return hipErrorNotSupported;
    const auto entry = bf16 ? (nn ? &gemm_silu_mul_layout<bf16_t, MI355_GEMM_NN> : &gemm_silu_mul_layout<bf16_t, MI355_GEMM_NT>)
                            : (nn ? &gemm_silu_mul_layout<half_t, MI355_GEMM_NN> : &gemm_silu_mul_layout<half_t, MI355_GEMM_NT>);
    return entry(A, B, C, M, N2, K, lda, ldb, ldc, variant, stream);
}

hipError_t gemm_step_qkv_dispatch(const void* x, const NormPrologue& norm, const void* w, void* qkv, int M, int N, int K, const RopeEpilogue& rope,
                                  int dtype, hipStream_t stream) {
    const auto entry = dtype == MI355_DTYPE_BF16 ? &gemm_step_qkv<bf16_t> : &gemm_step_qkv<half_t>;
    return entry(x, norm, w, qkv, M, N, K, K, K, N, rope, stream);
}

hipError_t gemm_step_gate_up_dispatch(const void* x, const NormPrologue& norm, const void* w, void* out, int M, int N, int K, int dtype,
                                      hipStream_t stream) {
    const auto entry = dtype == MI355_DTYPE_BF16 ? &gemm_step_gate_up<bf16_t> : &gemm_step_gate_up<half_t>;
    return entry(x, norm, w, out, M, N, K, K, K, N / 2, stream);
}

#ifdef MI355_TIMELINE
hipError_t (*timeline_hgemm_reader)(void*, size_t) = nullptr;
#endif

}  // namespace mi355

#ifdef MI355_TIMELINE
// profiling build: copies the records of the last tiled GEMM launch (kMaxWorkgroups x kSlots 64-bit values) to the host
extern "C" int mi355_timeline_read_hgemm(void* dst, size_t bytes) {
    return mi355::timeline_hgemm_reader ? (int)mi355::timeline_hgemm_reader(dst, bytes) : (int)hipErrorNotReady;
}
#endif
