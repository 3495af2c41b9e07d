// One call per forward pass of llama_layer.FineLlamaDecoderLayer: the eight launches of the layer (down to five for up to 8 rows) issued
// back to back from C++ through the C ABI of libmi355_serving.so. Issued one by one from Python (ctypes calls, tensor views, one
// allocation per intermediate) eight take the host ~85-95 us per layer, longer than a generation step keeps the GPU busy on any
// layer narrower than ~4096; from here ~25 us, with one block of torch's allocator for the intermediates: a step of one
// sequence through a layer 1024 wide 81 -> 29 us, 4 sequences through one 2048 wide 87 -> 45, first pass on new
// tensors 132 -> 61. With five launches the first of these takes 23 us, the second 41.
//
// Stateless: every tensor is an argument of the call, nothing is kept between calls.
#include <torch/extension.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <cmath>
#include <tuple>
#include <vector>

#include "mi355_serving.h"

// of the same library (csrc/mi355_serving_internal.h)
extern "C" size_t mi355_internal_gemm_copy_bytes(const void* A, const void* B, int M, int N, int K, int64_t lda, int64_t ldb, int layout);
extern "C" int mi355_internal_step_qkv(const void* x, const void* norm_weight, float eps, const void* w_qkv, void* qkv, void* kv_out, int B, int S,
                                       int q_heads, int kv_heads, int hidden, int64_t out_batch, int64_t out_row, int64_t out_head,
                                       const float* cos_table, const float* sin_table, const int32_t* positions, int64_t pos_batch, int n_positions,
                                       int dtype, void* stream);
extern "C" int mi355_internal_step_gate_up(const void* x, const void* norm_weight, float eps, const void* w_gu, void* out, int rows, int inter,
                                           int hidden, int dtype, void* stream);

namespace {

void check(int rc, const char* what) {
    TORCH_CHECK(rc == 0, what, ": ", mi355_last_error(), " (code ", rc, ")");
}

#define CHECK_HIP(expr)                                                         \
    do {                                                                        \
        const hipError_t err_ = (expr);                                         \
        TORCH_CHECK(err_ == hipSuccess, #expr ": ", hipGetErrorString(err_));   \
    } while (0)

struct Events {   // the pair of events around the attention block when it is timed
    hipEvent_t begin = nullptr, end = nullptr;
    ~Events() {
        if (begin) (void)hipEventDestroy(begin);
        if (end) (void)hipEventDestroy(end);
    }
};

// C = A W^T (+ R) for activations [M, K] and an nn.Linear weight [N, K], both with rows side by side
void linear(const void* a, const at::Tensor& w, const void* r, void* c, int64_t M, int dtype, hipStream_t stream) {
    const int64_t N = w.size(0), K = w.size(1);
    size_t need = mi355_internal_gemm_copy_bytes(a, w.data_ptr(), (int)M, (int)N, (int)K, K, K, MI355_GEMM_NT);
    at::Tensor ws;
    if (need > 0) {
        try {
            ws = at::empty({static_cast<int64_t>(need)}, w.options().dtype(at::kByte));
        } catch (const c10::OutOfMemoryError&) {
            need = 0;   // the product runs without aligned copies
        }
    }
    check(mi355_gemm_ws(a, w.data_ptr(), r, c, (int)M, (int)N, (int)K, K, K, N, N, MI355_GEMM_NT, dtype,
                        need > 0 ? ws.data_ptr() : nullptr, need, stream), "mi355_gemm_ws");
}

// hidden_states [B, S, H] -> (layer output [B, S, H], milliseconds of the attention block if `timed`, else 0). `positions`:
// int32, [S] for all batch rows or [B, S]. `kv`: empty without a cache; {cache} for a tensor [B, 2 n_kv, max_len, 128], whose rows
// past .. past + S - 1 are written; or {rows, k, v} for a cache of any layout: the [B, S, 2 n_kv, 128] view of the new tokens,
// which are written, and the [B, past + S or more, n_kv, 128] views of all keys and values. `gate_up_block`: 32 when w_gu alternates 32 gate rows with their 32 up rows, 0 when all
// gate rows precede all up rows.
std::tuple<at::Tensor, double> layer_forward(const at::Tensor& hidden_states, const at::Tensor& w_qkv, const at::Tensor& w_o,
                                             const at::Tensor& w_gu, const at::Tensor& w_d, const at::Tensor& ln1, const at::Tensor& ln2,
                                             const at::Tensor& cos, const at::Tensor& sin, const at::Tensor& positions, int64_t first_position,
                                             const std::vector<at::Tensor>& kv, int64_t past, int64_t n_q, int64_t n_kv, double eps,
                                             int64_t gate_up_block, bool timed) {
    constexpr int64_t D = 128;
    TORCH_CHECK(hidden_states.dim() == 3 && hidden_states.is_cuda(), "hidden_states must be a [B, S, H] GPU tensor");
    const int64_t B = hidden_states.size(0), S = hidden_states.size(1), H = hidden_states.size(2), rows = B * S;
    const auto type = hidden_states.scalar_type();
    TORCH_CHECK(type == at::kHalf || type == at::kBFloat16, "hidden_states must be float16 or bfloat16, got ", type);
    const bool bf16 = type == at::kBFloat16;
    const int dtype = bf16 ? MI355_DTYPE_BF16 : MI355_DTYPE_FP16;
    const int64_t heads = n_q + 2 * n_kv, F = w_d.size(1);
    TORCH_CHECK(B >= 1 && S >= 1 && rows <= INT32_MAX, "empty or too large hidden_states");
    const auto weight = [&](const at::Tensor& t, int64_t r, int64_t c, const char* name) {
        TORCH_CHECK(t.is_cuda() && t.device() == hidden_states.device() && t.scalar_type() == type && t.is_contiguous() && t.dim() == 2 &&
                    t.size(0) == r && t.size(1) == c, name, " must be a contiguous [", r, ", ", c, "] tensor of the hidden states' type and device");
    };
    weight(w_qkv, heads * D, H, "w_qkv");
    weight(w_o, H, n_q * D, "w_o");
    weight(w_gu, 2 * F, H, "w_gu");
    weight(w_d, H, F, "w_d");
    for (const at::Tensor* t : {&ln1, &ln2})
        TORCH_CHECK(t->is_cuda() && t->device() == hidden_states.device() && t->scalar_type() == type && t->is_contiguous() && t->numel() == H,
                    "norm weights must have the width, type and device of the hidden states");
    TORCH_CHECK(cos.is_cuda() && sin.is_cuda() && cos.scalar_type() == at::kFloat && sin.scalar_type() == at::kFloat && cos.is_contiguous() &&
                sin.is_contiguous() && cos.dim() == 2 && cos.size(1) == D / 2 && cos.sizes() == sin.sizes(), "cos and sin must be [n_positions, 64] float32");
    TORCH_CHECK(positions.is_cuda() && positions.scalar_type() == at::kInt && positions.is_contiguous() && first_position >= 0,
                "positions must be a contiguous int32 GPU tensor");
    // first_position > 0 or more entries than tokens: a window of S entries of a longer table
    const bool per_row = B > 1 && first_position == 0 && positions.numel() == rows && positions.dim() == 2;
    TORCH_CHECK(per_row || first_position + S <= positions.numel(), "positions has ", positions.numel(), " entries, ", first_position + S, " are needed");

    const c10::hip::HIPGuardMasqueradingAsCUDA guard(hidden_states.device());
    hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
    const at::Tensor x = hidden_states.contiguous();
    const int32_t* pos = positions.data_ptr<int32_t>() + first_position;
    const int64_t pos_batch = per_row ? S : 0;
    const float* cos_p = cos.data_ptr<float>();
    const float* sin_p = sin.data_ptr<float>();
    const int n_pos = (int)cos.size(0);

    // one block for the intermediates: norm output, fused projection, attention output, activated MLP rows
    const auto slot = [](int64_t elements) { return (elements + 127) / 128 * 128; };
    const int64_t n_h = slot(rows * H), n_qkv = slot(rows * heads * D), n_attn = slot(rows * n_q * D), n_act = slot(rows * F);
    const at::Tensor block = at::empty({n_h + n_qkv + n_attn + n_act}, x.options());
    char* base = static_cast<char*>(block.data_ptr());
    char* h = base;
    char* qkv = h + 2 * n_h;
    char* attn = qkv + 2 * n_qkv;
    char* act = attn + 2 * n_attn;
    at::Tensor out = at::empty({B, S, H}, x.options());

    const auto norm = [&](const void* in, const at::Tensor& w) {
        const auto entry = bf16 ? &mi355_rmsnorm_bf16 : &mi355_rmsnorm;
        check(entry(in, nullptr, nullptr, w.data_ptr(), h, rows, (int)H, H, 0, 0, H, (float)eps, stream), "mi355_rmsnorm");
    };
    // attention operands read where they lie: q in the fused projection, k and v there or in the cache (batch, head, row strides)
    const int64_t row = heads * D;
    struct Rows {   // where a [B, tokens, heads, 128] operand lies: bytes are 2 per element
        char* ptr;
        int64_t batch, row, head;
    };
    int64_t keys = S;
    // of the new tokens, keys in front of values; without a cache they stay where the projection puts them
    Rows fresh = {qkv + 2 * n_q * D, S * row, row, D};
    Rows k = {qkv + 2 * n_q * D, S * row, row, D}, v = {k.ptr + 2 * n_kv * D, S * row, row, D};
    if (!kv.empty()) {
        keys = past + S;
        if (kv.size() == 1) {
            const at::Tensor& t = kv[0];
            TORCH_CHECK(t.is_cuda() && t.device() == x.device() && t.scalar_type() == type && t.dim() == 4 && t.size(0) == B && t.size(1) == 2 * n_kv &&
                        t.size(3) == D && t.stride(3) == 1 && past >= 0 && past + S <= t.size(2),
                        "the KV cache must be a [B, 2 * n_kv, max_len, 128] tensor of the hidden states' type and device with room for the new tokens");
            k = {static_cast<char*>(t.data_ptr()), t.stride(0), t.stride(2), t.stride(1)};
            v = {k.ptr + 2 * n_kv * k.head, k.batch, k.row, k.head};
            fresh = {k.ptr + 2 * past * k.row, k.batch, k.row, k.head};
        } else {
            TORCH_CHECK(kv.size() == 3 && past >= 0, "kv: nothing, the cache tensor, or (rows, k, v)");
            const auto view = [&](const at::Tensor& t, int64_t tokens, int64_t n, const char* name) {
                TORCH_CHECK(t.is_cuda() && t.device() == x.device() && t.scalar_type() == type && t.dim() == 4 && t.size(0) == B && t.size(1) >= tokens &&
                            t.size(2) == n && t.size(3) == D && t.stride(3) == 1, "the KV cache's ", name, " must be a [", B, ", ", tokens, ", ", n,
                            ", 128] view of the hidden states' type and device");
                return Rows{static_cast<char*>(t.data_ptr()), t.stride(0), t.stride(1), t.stride(2)};
            };
            fresh = view(kv[0], S, 2 * n_kv, "new rows");
            k = view(kv[1], keys, n_kv, "keys");
            v = view(kv[2], keys, n_kv, "values");
        }
    }
    // Norm, projection and rotary embedding of up to 8 rows are one launch where their norm pays inside the product (norm_fits in
    // hgemm.hip), two where it does not, where the attention block is timed, which begins behind it, and of up to 64 rows whose
    // projection is the small-M kernel's; three otherwise.
    const auto step_qkv = [&](const void* in, const void* norm_weight) {
        if (rows > 64) return false;
        const int rc = mi355_internal_step_qkv(in, norm_weight, (float)eps, w_qkv.data_ptr(), qkv, fresh.ptr, (int)B, (int)S, (int)n_q, (int)n_kv, (int)H,
                                               fresh.batch, fresh.row, fresh.head, cos_p, sin_p, pos, pos_batch, n_pos, dtype, stream);
        if (rc != MI355_ERR_UNSUPPORTED) check(rc, "mi355_internal_step_qkv");
        return rc == 0;
    };
    Events ev;
    if (timed || rows > 8 || !step_qkv(x.data_ptr(), ln1.data_ptr())) {
        norm(x.data_ptr(), ln1);
        if (timed) {
            CHECK_HIP(hipEventCreate(&ev.begin));
            CHECK_HIP(hipEventCreate(&ev.end));
            CHECK_HIP(hipDeviceSynchronize());
            CHECK_HIP(hipEventRecord(ev.begin, stream));
        }
        if (!step_qkv(h, nullptr)) {
            linear(h, w_qkv, nullptr, qkv, rows, dtype, stream);
            if (kv.empty()) {
                const auto entry = bf16 ? &mi355_rope_bf16 : &mi355_rope;
                check(entry(qkv, qkv, (int)B, (int)S, (int)(n_q + n_kv), 0, (int)D, S * row, row, S * row, row, cos_p, sin_p, pos, pos_batch, n_pos,
                            stream), "mi355_rope");
            } else {
                const auto entry = bf16 ? &mi355_rope_qkv_bf16 : &mi355_rope_qkv;
                check(entry(qkv, fresh.ptr, (int)B, (int)S, (int)n_q, (int)n_kv, (int)D, S * row, row, fresh.batch, fresh.row, fresh.head, cos_p,
                            sin_p, pos, pos_batch, n_pos, stream), "mi355_rope_qkv");
            }
        }
    }
    {
        const int64_t strides[12] = {S * row, D, row, k.batch, k.head, k.row, v.batch, v.head, v.row, S * n_q * D, D, n_q * D};
        const auto entry = bf16 ? &mi355_fmha_fwd_bf16 : &mi355_fmha_fwd_strided;
        check(entry(qkv, k.ptr, v.ptr, attn, nullptr, (int)B, (int)n_q, (int)n_kv, (int)S, (int)keys, (int)D, 1.0f / std::sqrt((float)D), 1, (int)keys,
                    strides, stream), "mi355_fmha_fwd");
    }
    linear(attn, w_o, x.data_ptr(), out.data_ptr(), rows, dtype, stream);   // x + o_proj(attn)
    double ms = 0.0;
    if (timed) {
        float elapsed = 0.f;
        CHECK_HIP(hipEventRecord(ev.end, stream));
        CHECK_HIP(hipDeviceSynchronize());
        CHECK_HIP(hipEventElapsedTime(&elapsed, ev.begin, ev.end));
        ms = elapsed;
    }
    int rc = MI355_ERR_UNSUPPORTED;
    if (gate_up_block > 0 && rows <= 8) {
        rc = mi355_internal_step_gate_up(out.data_ptr(), ln2.data_ptr(), (float)eps, w_gu.data_ptr(), act, (int)rows, (int)F, (int)H, dtype, stream);
        if (rc != MI355_ERR_UNSUPPORTED) check(rc, "mi355_internal_step_gate_up");
    }
    const bool normalised = rc == 0;
    if (!normalised) norm(out.data_ptr(), ln2);
    if (!normalised && gate_up_block > 0) {
        const auto entry = bf16 ? &mi355_gemm_silu_mul_bf16 : &mi355_hgemm_silu_mul;
        rc = entry(h, w_gu.data_ptr(), act, (int)rows, (int)F, (int)H, H, H, F, MI355_GEMM_NT, stream);
        if (rc != MI355_ERR_UNSUPPORTED) check(rc, "mi355_hgemm_silu_mul");
    }
    if (rc == MI355_ERR_UNSUPPORTED) {   // shapes without the fused epilogue: the product, then the activation
        const at::Tensor gu = at::empty({rows, 2 * F}, x.options());
        linear(h, w_gu, nullptr, gu.data_ptr(), rows, dtype, stream);
        const auto entry = bf16 ? &mi355_silu_mul_bf16 : &mi355_silu_mul;
        check(entry(gu.data_ptr(), act, rows, (int)F, (int)gate_up_block, 2 * F, F, stream), "mi355_silu_mul");
    }
    linear(act, w_d, out.data_ptr(), out.data_ptr(), rows, dtype, stream);   // out + down_proj(act), in place
    return {out, ms};
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("layer_forward", &layer_forward, py::call_guard<py::gil_scoped_release>());
}
