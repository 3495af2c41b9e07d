// Host side of the GEMM entry points: aligned copies of operands, the choice of the translation unit that holds the kernels
// of an element type and layout (hgemm.hip), and the workspace of the split-K path.
#include <map>
#include <mutex>
#include <utility>
#include "mi355_common.h"
#include "mi355_serving_internal.h"

namespace mi355 {

static __global__ void hgemm_clear_kernel(unsigned* p, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0u;
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
        e = hipMalloc(&fresh_buf, want);
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

// An operand with unaligned rows is worth an aligned copy from a few K steps on: below that the bounds-checked kernel is
// done before a second launch would start.
size_t hgemm_workspace_bytes(const void* A, const void* B, int M, int N, int K, long lda, long ldb, int layout) {
    if (K <= 64) return 0;
    const GemmPackPlan plan = gemm_pack_plan(A, B, M, N, K, lda, ldb, layout);
    return plan.a.pack || plan.b.pack ? plan.bytes() : 0;
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
    if (const size_t need = workspace ? hgemm_workspace_bytes(A, B, M, N, K, lda, ldb, layout) : 0; need > 0 && need <= workspace_bytes) {
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
