// Aligned copies of GEMM operands whose rows are not 16-byte aligned (a dense matrix whose row length is not a multiple of
// 8, a view that starts at an odd element). The tiled kernels' global -> LDS copies move 16 aligned bytes; the direct kernel
// (hgemm_direct.hip) reads such operands where they lie, at about half the tiled kernels' rate on large products. Which of the two a
// product takes: copies_pay in hgemm_dispatch.hip, with both sides measured.
#include "mi355_common.h"
#include "mi355_serving_internal.h"

namespace mi355 {
namespace {

// rows x cols 16-bit elements at src (row stride ld, any alignment) -> dst, rows of `chunks` 16-byte chunks; the elements
// behind a row's end are zero
struct PackJob {
    const uint16_t* src;
    uint16_t* dst;
    long ld;
    int cols;
    uint32_t chunks, total;   // chunks per row, chunks in all
};

constexpr int kPackThreads = 256;
constexpr int kPackPerThread = 4;   // chunks of a thread, all of them in flight together

// Bandwidth-bound: one read and one write of the operand. A thread moves 16-byte chunks (consecutive threads consecutive
// chunks); the reads are 16-byte loads of no stated alignment, which global memory takes at any element.
__global__ __launch_bounds__(kPackThreads) void gemm_pack_kernel(PackJob a, PackJob b, uint32_t blocks_a) {
    const bool second = blockIdx.x >= blocks_a;
    const PackJob& job = second ? b : a;
    const uint32_t first = (second ? blockIdx.x - blocks_a : blockIdx.x) * (kPackThreads * kPackPerThread) + threadIdx.x;
    int4v v[kPackPerThread];
#pragma unroll
    for (int u = 0; u < kPackPerThread; ++u) {
        const uint32_t i = first + u * kPackThreads;
        v[u] = int4v{0, 0, 0, 0};
        if (i >= job.total) continue;
        const uint32_t row = i / job.chunks;
        const int col = (int)(i - row * job.chunks) * 8;
        const uint16_t* p = job.src + (long)row * job.ld + col;
        if (col + 8 <= job.cols) {
            __builtin_memcpy(&v[u], p, 16);
        } else {
            uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (col + j < job.cols) w[j >> 1] |= (uint32_t)p[j] << (16 * (j & 1));
            v[u] = int4v{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
        }
    }
#pragma unroll
    for (int u = 0; u < kPackPerThread; ++u) {
        const uint32_t i = first + u * kPackThreads;
        if (i < job.total) *(int4v*)(job.dst + (long)i * 8) = v[u];
    }
}

PackJob job_of(const void* src, void* dst, long ld, const GemmPackPlan::Operand& op) {
    PackJob j;
    j.src = static_cast<const uint16_t*>(src);
    j.dst = static_cast<uint16_t*>(dst);
    j.ld = ld;
    j.cols = op.cols;
    j.chunks = (uint32_t)(op.ld / 8);
    j.total = op.pack ? (uint32_t)(op.bytes / 16) : 0u;
    return j;
}

}  // namespace

GemmPackPlan gemm_pack_plan(const void* A, const void* B, int M, int N, int K, long lda, long ldb, int layout) {
    GemmPackPlan p;
    const bool a_kc = layout != MI355_GEMM_TN, b_kc = layout == MI355_GEMM_NT;
    const auto operand = [](const void* ptr, long ld, int rows, int cols) {
        GemmPackPlan::Operand op;
        op.cols = cols;
        op.pack = reinterpret_cast<uintptr_t>(ptr) % 16 != 0 || ld % 8 != 0;
        op.ld = op.pack ? ((long)cols + 7) / 8 * 8 : ld;
        op.bytes = op.pack ? (size_t)op.ld * rows * 2 : 0;
        return op;
    };
    p.a = operand(A, lda, a_kc ? M : K, a_kc ? K : M);
    p.b = operand(B, ldb, b_kc ? N : K, b_kc ? K : N);
    // the kernels that read the copies address rows of up to 2^22 elements; chunks are counted in 32 bits
    if (p.a.ld >= (1L << 22) || p.b.ld >= (1L << 22) || p.a.bytes / 16 >= (size_t(1) << 31) || p.b.bytes / 16 >= (size_t(1) << 31))
        p.a.pack = p.b.pack = false;
    if (!p.a.pack && !p.b.pack) p.a.bytes = p.b.bytes = 0;
    return p;
}

hipError_t gemm_pack_launch(const GemmPackPlan& p, const void* A, const void* B, long lda, long ldb, void* a_copy, void* b_copy, hipStream_t stream) {
    const PackJob ja = job_of(A, a_copy, lda, p.a), jb = job_of(B, b_copy, ldb, p.b);
    constexpr uint32_t kPerBlock = kPackThreads * kPackPerThread;
    const uint32_t blocks_a = (ja.total + kPerBlock - 1) / kPerBlock, blocks_b = (jb.total + kPerBlock - 1) / kPerBlock;
    gemm_pack_kernel<<<dim3(blocks_a + blocks_b), dim3(kPackThreads), 0, stream>>>(ja, jb, blocks_a);
    return hipGetLastError();
}

}  // namespace mi355
