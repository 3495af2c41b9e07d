// Decode-shaped attention forward for gfx950 (MI355X): few query rows per kv head, any number of keys.
//
// The reference runs its generation step (`is_decode`, one query row padded to 64 by ops.py:19-25) through the
// prefill kernel, one workgroup per (batch, q head) walking all keys (semi/fmha_2_amd.cpp:341-356); that leaves
// almost the whole GPU idle and is bound by one workgroup's memory rate. Here the step is a split-KV
// ("flash-decoding") pass in ONE launch, HBM-bound by the single read of K and V:
//
//   * a workgroup = (batch, kv head, key range); about one workgroup per CU or, where that is expected to be done sooner, up to
//     two rounds of them (decode_plan). The query rows of all q heads that share
//     the kv head are packed side by side as the (up to 32) columns of the S^T = K Q^T product, so K and V are read once
//     per kv head, not once per q head.
//   * the waves of a workgroup cut its key range into contiguous pieces; each wave streams its piece in tiles of 32 keys
//     through a private LDS pipeline (direct-to-LDS copies, no workgroup barriers while streaming) and runs the
//     register-resident online softmax of the prefill kernel.
//   * the waves' results are combined through LDS and written as one unnormalised partial result per workgroup
//     (O~ [128], m, l per column, fp32) to a workspace; the workgroup then takes a ticket from a counter of its
//     (batch, kv head), and the one that draws the last ticket combines all partials of that pair,
//     O = sum_s 2^((m_s - m) c) O~_s / sum_s 2^((m_s - m) c) l_s, writes O and LSE and puts the counter back to zero.
//     With a single key range per (batch, kv head) the workgroup writes O and LSE directly and touches no workspace.
//
// Mask semantics are those of the prefill kernel (keys >= kv_valid_len masked; causal: key j visible to query i
// iff j <= i + Sk - Sq).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <map>
#include <mutex>
#include <utility>

#include "mi355_common.h"
#include "mi355_serving_internal.h"
#include "mi355_timeline.h"

namespace mi355 {

// profiling build: per workgroup, wall clock at [entry, first tile landed, key range done, partial results stored, ticket
// drawn, merge: partial results landed, merge: summed, exit] (0 = the workgroup did not get there)
MI355_TL(static __device__ unsigned long long fmha_decode_stamps[timeline::kMaxWorkgroups * timeline::kSlots];)

namespace dec {
constexpr int D = 128;
constexpr int TK = 32;                       // keys per tile
constexpr int ROW_BYTES = D * 2;             // 256
constexpr int TILE_BYTES = TK * ROW_BYTES;   // 8 KiB
constexpr int STAGE_BYTES = 2 * TILE_BYTES;  // K + V
constexpr float kLazyLog2 = 8.f;             // rescale only when a column maximum grows by more than 2^8
constexpr int COPIES = 2 * (TILE_BYTES / 1024);  // 16 copy instructions per stage
constexpr int PART_STRIDE = D + 4;           // floats per (workgroup, column): O~[128], m, l, 2 pad (keeps rows 16-byte aligned)
// Ticket counters lie this many 32-bit words (256 bytes) apart. Device-scope atomics of workgroups on different XCDs are
// carried out at the memory side, one after the other per address range: with the counters of all (batch, kv head)
// pairs in one 64-byte line, the 256 tickets of a call queued up behind each other (~12 ns each, 3 us from the first to
// the last at batch 1); 256 bytes apart they proceed side by side (a larger stride brought nothing more).
constexpr int kCounterStride = 64;
// The counters occupy a region of FIXED size at the start of every workspace, whatever the call: a workspace is shared by
// calls of different shapes, each of which leaves its counters at zero, and a region that grew and shrank with the number
// of (batch, kv head) pairs would let one call's partial results land where the next call keeps its counters. A call is
// cut into several key ranges only while it has at most kMaxSplitPairs pairs.
constexpr int kMaxSplitPairs = 255;
constexpr size_t kCounterBytes = size_t(kMaxSplitPairs + 1) * kCounterStride * sizeof(unsigned);   // 64 KiB

__device__ __forceinline__ int swz_k(int row) { return row & 15; }
__device__ __forceinline__ int swz_v(int row) { return (row & 7) << 1; }
// maximum / sum over the four lanes that hold a column
__device__ __forceinline__ float quad_max(float x) {
    x = fmaxf(x, __shfl_xor(x, 16, 64));
    return fmaxf(x, __shfl_xor(x, 32, 64));
}
__device__ __forceinline__ float quad_sum(float x) {
    x += __shfl_xor(x, 16, 64);
    return x + __shfl_xor(x, 32, 64);
}
}  // namespace dec

// How a launch is dealt out: query heads per kv head, and the divisions a workgroup needs to find its part (1 x 32/8 heads over 8191 keys
// 12.3 us with divisions on the device, 12.2 so)
struct DecodeMap {
    int group;
    Divisor by_splits, by_hkv, by_sq;
};

// Workgroup wg = (b * Hkv + hkv) * splits + s covers key tiles [s * tiles_per_split, (s + 1) * tiles_per_split).
// WAVES waves with NSTAGE pipeline stages of 16 KiB each (two waves: a single key range only). <4, 2> (one wave per SIMD, one tile in flight behind the one
// being consumed, 128 KiB of LDS) measured better than <3, 3> for short and for long key ranges alike.
// NB: blocks of 16 columns. Both products are MFMA 16x16x32, laid out as in the prefill kernel (fmha_fwd.hip): S^T[kb] (16 keys x 16 columns)
// = K[kb] Q^T, O^T[db] (16 d x 16 columns) += V^T[db] P^T; a lane holds 4 keys of a key block, or 4 d of a d block, of one column, the statistics
// of a column live in four lanes, which only talk to each other when the exponent reference moves. A wave is alone on its SIMD and a tile a
// chain of dependent steps: with 32x32x16 instructions, eight of them one behind the other for S^T, half of their columns empty where a kv
// head has up to 16 query rows, and a cross-lane maximum in every tile, 301 keys (three tiles a wave) of 1 x 8/2 heads took 7.2 us, now 5.9;
// the combine of the waves, then one output and two exponentials per thread and column, is part of that (1.4 -> 0.9 us). 1 x 32/8 heads over 256
// keys 6.3 -> 5.1, 500 8.5 -> 7.0, 8191 12.8 -> 12.2, 64 x 64/8 over 300 19.8 -> 16.9; 8 x 32/8 over 8192, bound by HBM, 50.6 either way.
template <typename T, int WAVES, int NSTAGE, int NB>
__global__ __launch_bounds__(WAVES * 64) void fmha_decode_kernel(
    const T* __restrict__ Q, const T* __restrict__ K, const T* __restrict__ V, T* __restrict__ O, float* __restrict__ LSE,
    float* part, unsigned* counters, int B, int Hq, int Hkv, int Sq, int Sk, float scale_log2, int causal, int kv_valid,
    int splits, int tiles_per_split, FmhaStrides sd, DecodeMap map) {
    using namespace dec;
    using V8 = typename Elem<T>::v8;
    MI355_TL(unsigned long long tl[8] = {timeline::wall_clock(), 0, 0, 0, 0, 0, 0, 0};
             auto tl_dump = [&]() {
                 if (threadIdx.x == 0 && blockIdx.x < timeline::kMaxWorkgroups)
                     for (int i = 0; i < 8; ++i) fmha_decode_stamps[(long)blockIdx.x * timeline::kSlots + i] = tl[i];
             };)
    constexpr int WAVE_BYTES = NSTAGE * STAGE_BYTES;
    constexpr int NTHREADS = WAVES * 64;
    extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    MI355_LDS char* wbase = (MI355_LDS char*)smem_raw + wave * WAVE_BYTES;

    const int g = lane >> 4;
    const int c16 = lane & 15;
    const int bh = divide(blockIdx.x, map.by_splits);
    const int s_idx = blockIdx.x - bh * splits;
    const int b = divide(bh, map.by_hkv);
    const int hkv = bh - b * Hkv;
    const int group = map.group;
    const int ncols = group * Sq;  // <= 16 NB
    const int shift = Sk - Sq;

    const T* Kh = K + b * sd.k_batch + hkv * sd.k_head;
    const T* Vh = V + b * sd.v_batch + hkv * sd.v_head;

    // this workgroup's tiles, and this wave's contiguous piece of them (possibly empty)
    const int tiles = (kv_valid + TK - 1) / TK;
    const int g_begin = s_idx * tiles_per_split;
    const int g_end = min(g_begin + tiles_per_split, tiles);
    const int per_wave = (max(g_end - g_begin, 0) + WAVES - 1) / WAVES;
    const int t_begin = min(g_begin + wave * per_wave, g_end);
    const int t_end = min(t_begin + per_wave, g_end);

    // copy i (0..7) of a tile covers rows 4i + lane/16, chunk position lane%16; addresses = wave-uniform tile base (scalar
    // registers) + 32-bit lane offset; rows past the last valid key are clamped onto it (masked later, but V must not
    // feed NaNs into 0 * V)
    const int c_row = lane >> 4;
    const uint32_t k_row_bytes = (uint32_t)sd.k_row * 2, v_row_bytes = (uint32_t)sd.v_row * 2;
    const uint32_t kcol = (lane & 15);
    auto issue_stage = [&](int tile, int slot) {
        MI355_LDS char* st = wbase + slot * STAGE_BYTES;
        const int tile_u = __builtin_amdgcn_readfirstlane(tile);
        const char* kb = (const char*)Kh + (long)tile_u * TK * sd.k_row * 2;
        const char* vb = (const char*)Vh + (long)tile_u * TK * sd.v_row * 2;
        const int last = kv_valid - 1 - tile_u * TK;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            int row = 4 * i + c_row;
            copy16_global_to_lds(kb, (uint32_t)min(row, last) * k_row_bytes + ((kcol ^ swz_k(row)) << 4), st + i * 1024);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            int row = 4 * i + c_row;
            copy16_global_to_lds(vb, (uint32_t)min(row, last) * v_row_bytes + ((kcol ^ swz_v(row)) << 4),
                                 st + TILE_BYTES + i * 1024);
        }
    };

    const int k_base = c16 * ROW_BYTES + ((g ^ c16) << 4);   // xor (ks << 6), + kb * 16 rows
    const int v_row = 4 * g + (c16 >> 2);
    const int v_base = TILE_BYTES + v_row * ROW_BYTES + ((((c16 & 3) >> 1) ^ swz_v(v_row)) << 4) + (c16 & 1) * 8;  // xor (db << 5)

    float4v o[NB][8];
    float m_run[NB], l_run[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        m_run[nb] = -INFINITY;
        l_run[nb] = 0.f;
#pragma unroll
        for (int db = 0; db < 8; ++db) o[nb][db] = float4v{0.f, 0.f, 0.f, 0.f};
    }

    const int n_loc = t_end - t_begin;
    // each wave starts at a different tile of its piece and wraps around (the online softmax does not care about the
    // order): waves whose pieces lie a large power of two apart then do not walk the same memory channels in step
    const int rot = n_loc > 0 ? ((blockIdx.x * WAVES + wave) * 5) % n_loc : 0;
    auto tile_of = [&](int i) { int r = i + rot; return t_begin + (r >= n_loc ? r - n_loc : r); };
    int issued = t_begin;
#pragma unroll
    for (int i = 0; i < NSTAGE - 1; ++i)
        if (issued < t_end) {
            issue_stage(tile_of(issued - t_begin), i);
            ++issued;
        }
    // Everything about the queries comes behind the first key / value copies, so that those leave as early as possible
    // and the latency of the query fetch hides under theirs.
    // column c of the packed query block = (q head hkv*group + c / Sq, query row c % Sq)
    int lim[NB];      // last visible key of this lane's column(s)
    V8 qf[NB][4];     // Q[column][32 ks + 8 g .. +7]
    int lim_min = kv_valid - 1;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int col = min(16 * nb + c16, ncols - 1);
        const int head = divide(col, map.by_sq);
        const int hq = hkv * group + head;
        const int qi = col - head * Sq;
        const T* qp = Q + b * sd.q_batch + hq * sd.q_head + qi * sd.q_row + 8 * g;
        lim[nb] = causal ? min(kv_valid - 1, qi + shift) : kv_valid - 1;
        lim_min = min(lim_min, lim[nb]);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) qf[nb][ks] = *(const V8*)(qp + ks * 32);
    }
    // smallest such limit over the wave: tiles that end at or before it need no mask code
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) lim_min = min(lim_min, __shfl_xor(lim_min, off, 64));
    lim_min = __builtin_amdgcn_readfirstlane(lim_min);
    // A use of the query fragments in front of the loop: the compiler waits for their loads where they are first used,
    // and it does not count the tile copies (inline assembly) among the loads in flight. With the first use inside the
    // loop that wait, "everything I know of has landed", came back on every iteration as vmcnt(0) in front of the S^T
    // products and held each tile's arithmetic until the NEXT tile's copies had landed too: no copy ever overlapped
    // arithmetic. Out here it waits once, for the first tile and the queries, which the first iteration needs anyway.
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) asm volatile("" : "+v"(qf[nb][0]), "+v"(qf[nb][1]), "+v"(qf[nb][2]), "+v"(qf[nb][3]));
    int slot = 0, fill = NSTAGE - 1;
    for (int tt0 = t_begin; tt0 < t_end; ++tt0) {
        const int t = tile_of(tt0 - t_begin);
        if (issued < t_end) {
            issue_stage(tile_of(issued - t_begin), fill);
            ++issued;
            fill = (fill + 1 == NSTAGE) ? 0 : fill + 1;
            wait_vmcnt<COPIES*(NSTAGE - 1)>();  // everything but the newest NSTAGE-1 tiles has landed
        } else {
            wait_vmcnt<0>();
        }
        MI355_TL(if (tt0 == t_begin) tl[1] = timeline::wall_clock();)
        MI355_LDS char* st = wbase + slot * STAGE_BYTES;
        slot = (slot + 1 == NSTAGE) ? 0 : slot + 1;

        // S^T = K Q^T: lane holds keys 16 kb + 4 g + 0..3 of its column
        float4v s[NB][2];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) s[nb][0] = s[nb][1] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                V8 kf = Elem<T>::frag(lds_read_b128(st + ((k_base ^ (ks << 6)) + kb * 16 * ROW_BYTES)));
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) s[nb][kb] = Elem<T>::mfma16(kf, qf[nb][ks], s[nb][kb]);
            }
        const int key0 = t * TK;
        if (key0 + TK - 1 > lim_min) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (key0 + 16 * (e >> 2) + 4 * g + (e & 3) > lim[nb]) s[nb][e >> 2][e & 3] = -INFINITY;
        }
        // lazy rescaling as in the prefill kernel: m_run is the exponent reference of the running sums and only moves
        // (with O and l rescaled) when some score exceeds it by more than 2^kLazyLog2
        float mx[NB];
        bool raise = false;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            mx[nb] = fmaxf(fmaxf(fmaxf(s[nb][0][0], s[nb][0][1]), fmaxf(s[nb][0][2], s[nb][0][3])),
                           fmaxf(fmaxf(s[nb][1][0], s[nb][1][1]), fmaxf(s[nb][1][2], s[nb][1][3])));
            raise = raise || (mx[nb] - m_run[nb]) * scale_log2 > kLazyLog2;  // -inf - -inf = NaN compares false
        }
        if (__builtin_amdgcn_ballot_w64(raise) != 0) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const float m_new = fmaxf(m_run[nb], quad_max(mx[nb]));
                const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
                const float alpha = __builtin_amdgcn_exp2f((m_run[nb] - m_use) * scale_log2);
                m_run[nb] = m_new;
                l_run[nb] *= alpha;
#pragma unroll
                for (int db = 0; db < 8; ++db) o[nb][db] *= alpha;
            }
        }
        V8 pf[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const float neg_ms = (m_run[nb] == -INFINITY) ? 0.f : -m_run[nb] * scale_log2;
            float psum = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[nb][e >> 2][e & 3], scale_log2, neg_ms));
                psum += p;
                pf[nb][e] = (T)p;
            }
            l_run[nb] += psum;
        }
        // O^T += V^T P^T; the 8 keys of a lane of P are 4 g + 0..3 and 16 + 4 g + 0..3, V^T is gathered in that order
#pragma unroll
        for (int db = 0; db < 8; ++db) {
            MI355_LDS char* vp = st + (v_base ^ (db << 5));
            V8 vf = Elem<T>::frag(concat(lds_read_tr16_b64(vp), lds_read_tr16_b64(vp + 16 * ROW_BYTES)));
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) o[nb][db] = Elem<T>::mfma16(vf, pf[nb], o[nb][db]);
        }
        wait_lgkmcnt<0>();  // the reads of this slot are complete before a later copy refills it
    }

    // ---- combine the waves of the workgroup through LDS (the pipelines are drained: their memory is free) ------------
    // per wave: O~ [ncols][128] floats, then m [32], l [32]
    MI355_TL(tl[2] = timeline::wall_clock();)
    __syncthreads();
    MI355_LDS float* cmb = (MI355_LDS float*)smem_raw;
    const int wave_floats = ncols * D + 64;
    {
        MI355_LDS float* mine = cmb + wave * wave_floats;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int col = 16 * nb + c16;
            const float l_tot = quad_sum(l_run[nb]);
            if (col < ncols) {
#pragma unroll
                for (int db = 0; db < 8; ++db) *(MI355_LDS float4v*)(mine + col * D + db * 16 + 4 * g) = o[nb][db];
                if (g == 0) {
                    mine[ncols * D + col] = m_run[nb];
                    mine[ncols * D + 32 + col] = l_tot;
                }
            }
        }
    }
    __syncthreads();
    const long row0 = ((long)b * Hq + (long)hkv * group) * Sq;   // LSE index of column 0 (columns are consecutive rows)
    const int n_out = ncols * (D / 4);   // output elements f = (column f / 32, d 4 (f % 32) .. +3)
    // an output element over the workgroup's waves; weights 2^((m_w - m) c), 0 for waves without a visible key
    auto combined = [&](int f, float& m_out, float& l_out) {
        const int c = f >> 5;
        float mw[WAVES], lw[WAVES];
        float4v ow[WAVES];
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            mw[w] = cmb[w * wave_floats + ncols * D + c];
            lw[w] = cmb[w * wave_floats + ncols * D + 32 + c];
            ow[w] = *(MI355_LDS const float4v*)(cmb + w * wave_floats + 4 * f);
        }
        float m = -INFINITY, l = 0.f;
        float4v acc = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < WAVES; ++w) m = fmaxf(m, mw[w]);
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float wgt = (m == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f((mw[w] - m) * scale_log2);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] += wgt * ow[w][e];
            l += wgt * lw[w];
        }
        m_out = m;
        l_out = l;
        return acc;
    };
    auto store_out = [&](int f, const float4v& acc, float m, float l) {
        const int c = f >> 5, d = (f & 31) * 4;
        const float inv = (l > 0.f) ? 1.f / l : 0.f;
        const int head = divide(c, map.by_sq), chq = hkv * group + head, cqi = c - head * Sq;
        typename Elem<T>::v4 ov;
#pragma unroll
        for (int e = 0; e < 4; ++e) ov[e] = (T)(acc[e] * inv);
        *(typename Elem<T>::v4*)(O + b * sd.o_batch + chq * sd.o_head + cqi * sd.o_row + d) = ov;
        if (LSE != nullptr && d == 0)
            LSE[row0 + c] = (l > 0.f) ? (m * scale_log2 + __builtin_log2f(l)) * 0.69314718055994531f : -INFINITY;
    };
    if (splits == 1) {   // the only key range of this (batch, kv head): the result is final
        for (int f = tid; f < n_out; f += NTHREADS) {
            float m, l;
            const float4v acc = combined(f, m, l);
            store_out(f, acc, m, l);
        }
        MI355_TL(wait_vmcnt<0>(); tl[7] = timeline::wall_clock(); tl_dump();)
        return;
    }
    // Partial results cross XCDs (each has its own L2). The hand-over from the workgroups that write them to the one that
    // merges them is ordered by instructions, not by a release / acquire pair: a device-scope fence writes back and
    // invalidates a whole L2 here, and an acquire-release ticket costs 2.5-3 us per launch (b = 1 over 8192 keys: 13.8 us
    // against 11.0). What takes the fence's place, step by step:
    //   1. every partial result is stored with a device-scope atomic store, i.e. `global_store_dwordx2 .. sc1`: written through
    //      the XCD's L2 to memory, nothing of it stays dirty in a cache;
    //   2. `s_waitcnt vmcnt(0)` behind the stores: on gfx9-family parts a store leaves vmcnt only when the memory system has
    //      acknowledged it at the scope it was issued with. The wait is an assembly statement with a memory clobber, so the
    //      compiler keeps the stores in front of it;
    //   3. the workgroup barrier: all threads have passed their wait before thread 0 draws the ticket;
    //   4. the ticket is a device-scope atomic add, carried out at the memory side: the tickets of one counter are totally
    //      ordered, and the workgroup that draws the last one knows that every other workgroup of its (batch, kv head) has
    //      passed step 2;
    //   5. the merging workgroup reads the partial results with `global_load_dword[x4] .. sc1` (device-coherent: served from
    //      memory, not from a line its XCD's L2 may still hold from an earlier launch), issued behind the branch on the
    //      ticket's value, which the hardware cannot pass before the atomic has returned.
    // tests/test_inline_asm_loads_cpu.py checks 1, 2 and 5 in the generated code.
    float* mypart = part + (long)blockIdx.x * ncols * PART_STRIDE;
    for (int f = tid; f < n_out; f += NTHREADS) {
        const int c = f >> 5, d = (f & 31) * 4;
        float m, l;
        const float4v acc = combined(f, m, l);
        const auto pair = [](float x, float y) { return (uint64_t)__builtin_bit_cast(uint32_t, x) | (uint64_t)__builtin_bit_cast(uint32_t, y) << 32; };
        uint64_t* dst = reinterpret_cast<uint64_t*>(mypart + c * PART_STRIDE + d);
        __hip_atomic_store(dst, pair(acc[0], acc[1]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(dst + 1, pair(acc[2], acc[3]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (d == 0) __hip_atomic_store(reinterpret_cast<uint64_t*>(mypart + c * PART_STRIDE + D), pair(m, l), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // ---- ticket: the workgroup that completes the set of key ranges of (b, hkv) merges them ----------------------------
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this thread's partial results have reached memory before the ticket is drawn
    MI355_TL(tl[3] = timeline::wall_clock();)
    __syncthreads();
    MI355_LDS unsigned* ticket_sh = (MI355_LDS unsigned*)(cmb + WAVES * wave_floats);
    if (tid == 0) *ticket_sh = __hip_atomic_fetch_add(&counters[(long)bh * kCounterStride], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    MI355_TL(tl[4] = timeline::wall_clock();)
    if (*ticket_sh != (unsigned)(splits - 1)) {
        MI355_TL(tl[7] = tl[4]; tl_dump();)
        return;
    }
    // last ticket: every other workgroup of (b, hkv) drew its ticket after its partial results had reached memory.
    // They are read back with device-coherent loads (sc1), many in flight per thread: one memory round trip for the
    // statistics, then one per 16 key ranges for the outputs.
    const float* base = part + (long)bh * splits * ncols * PART_STRIDE;
    const long split_stride = (long)ncols * PART_STRIDE;
    MI355_LDS float* st_m = cmb;                          // [splits][ncols]: m_s
    MI355_LDS float* st_l = cmb + splits * ncols;         // [splits][ncols]: l_s
    constexpr int BATCH = 32;
    // BATCH loads of 16 bytes each: the outputs of key ranges sp0 .. sp0 + BATCH - 1 for 4 d of one column
    // (in groups of 8 key ranges, a group only when it holds a key range that exists: a call with 4 key ranges issues 8
    // loads per thread, not 32; within a group, key ranges past the last one repeat it and get weight zero)
    auto load_batch = [&](float4v(&v)[BATCH], const float* pc, int sp0, int sp_end) {
#pragma unroll
        for (int g8 = 0; g8 < BATCH; g8 += 8) {
            if (sp0 + g8 < sp_end) {
#pragma unroll
                for (int u = g8; u < g8 + 8; ++u) {
                    const float* pa = pc + (long)min(sp0 + u, sp_end - 1) * split_stride;
                    asm volatile("global_load_dwordx4 %0, %1, off sc1" : "=v"(v[u]) : "v"(pa) : "memory");
                }
            }
        }
    };
    auto wait_batch = [](float4v(&v)[BATCH]) {   // the loads above have landed; nothing that uses v moves in front of this
        asm volatile("s_waitcnt vmcnt(0)"
                     : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]), "+v"(v[8]),
                       "+v"(v[9]), "+v"(v[10]), "+v"(v[11]), "+v"(v[12]), "+v"(v[13]), "+v"(v[14]), "+v"(v[15])
                     :: "memory");
        asm volatile("" : "+v"(v[16]), "+v"(v[17]), "+v"(v[18]), "+v"(v[19]), "+v"(v[20]), "+v"(v[21]), "+v"(v[22]), "+v"(v[23]),
                          "+v"(v[24]), "+v"(v[25]), "+v"(v[26]), "+v"(v[27]), "+v"(v[28]), "+v"(v[29]), "+v"(v[30]), "+v"(v[31]));
    };
    // the first batch of this thread's first output element goes out before the statistics are fetched: one memory
    // round trip serves both
    float4v v[BATCH];
    // Where the outputs are a half or a quarter as many as the threads (or fewer), two or four threads share one and take a part of
    // the key ranges each; their sums meet in LDS, in order.
    const int parts = n_out * 4 <= NTHREADS ? 4 : n_out * 2 <= NTHREADS ? 2 : 1;
    const int per_part = (splits + parts - 1) / parts;
    const int my_part = parts == 1 ? 0 : tid / n_out;   // >= parts: an idle thread
    const int first_sp = my_part * per_part, end_sp = my_part < parts ? min(first_sp + per_part, splits) : first_sp;
    const int first_f = parts == 1 ? tid : tid - my_part * n_out;
    if (first_f < n_out && first_sp < end_sp) load_batch(v, base + (first_f >> 5) * PART_STRIDE + (first_f & 31) * 4, first_sp, end_sp);
    for (int i = tid; i < splits * ncols; i += NTHREADS) {
        const float* ps = base + (long)(i / ncols) * split_stride + (i % ncols) * PART_STRIDE + D;
        float ms, ls;
        asm volatile("global_load_dword %0, %2, off sc1\n\tglobal_load_dword %1, %2, off offset:4 sc1\n\ts_waitcnt vmcnt(0)"
                     : "=&v"(ms), "=&v"(ls) : "v"(ps) : "memory");
        st_m[i] = ms;
        st_l[i] = ls;
    }
    MI355_TL(tl[5] = timeline::wall_clock();)
    __syncthreads();
    // The weight of key range s for column c, 2^((m_s - m_c) scale), is worked out once, by thread s * ncols + c, and left in
    // LDS together with its share of the row sum; the accumulation loop below then is two LDS reads and four
    // multiply-adds per key range.
    MI355_LDS float* st_w = cmb + 2 * splits * ncols;     // [splits][ncols]: weight of key range s
    MI355_LDS float* st_mc = cmb + 3 * splits * ncols;    // [ncols]: m_c
    for (int i = tid; i < splits * ncols; i += NTHREADS) {
        const int c = i % ncols;
        float m = -INFINITY;
        for (int sp0 = 0; sp0 < splits; sp0 += 8) {   // 8 independent LDS reads at a time
            float ms[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) ms[u] = st_m[min(sp0 + u, splits - 1) * ncols + c];
#pragma unroll
            for (int u = 0; u < 8; ++u) m = fmaxf(m, ms[u]);
        }
        const float w = (m == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f((st_m[i] - m) * scale_log2);
        st_w[i] = w;
        st_l[i] *= w;
        if (i < ncols) st_mc[c] = m;
    }
    __syncthreads();
    MI355_LDS float* st_acc = cmb + ((3 * splits * ncols + ncols + 3) & ~3);   // [parts - 1][n_out][4], then [parts - 1][n_out]: their sums of l
    for (int f = first_f; f < n_out; f += NTHREADS) {   // (more than one part: every thread, once)
        const int c = f >> 5;
        const float* pc = base + c * PART_STRIDE + (f & 31) * 4;
        float4v acc = float4v{0.f, 0.f, 0.f, 0.f};
        float l = 0.f;
        for (int sp0 = first_sp; sp0 < end_sp; sp0 += BATCH) {
            if (f != first_f || sp0 != first_sp) load_batch(v, pc, sp0, end_sp);
            // the weights of this batch, while its loads are in flight (all LDS reads first, so they overlap each other);
            // key ranges past the last one repeat it with weight zero
            float wgt[BATCH], ls[BATCH];
#pragma unroll
            for (int g8 = 0; g8 < BATCH; g8 += 8) {
                if (sp0 + g8 < end_sp) {
#pragma unroll
                    for (int u = g8; u < g8 + 8; ++u) {
                        const int sp = min(sp0 + u, end_sp - 1);
                        wgt[u] = st_w[sp * ncols + c];
                        ls[u] = st_l[sp * ncols + c];
                    }
#pragma unroll
                    for (int u = g8; u < g8 + 8; ++u) {
                        if (sp0 + u >= end_sp) wgt[u] = ls[u] = 0.f;
                        l += ls[u];
                    }
                }
            }
            wait_batch(v);
#pragma unroll
            for (int g8 = 0; g8 < BATCH; g8 += 8) {
                if (sp0 + g8 < end_sp) {
#pragma unroll
                    for (int u = g8; u < g8 + 8; ++u)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[e] += wgt[u] * v[u][e];
                }
            }
        }
        if (parts > 1) {
            if (my_part > 0 && my_part < parts) {
                *(MI355_LDS float4v*)(st_acc + 4 * ((my_part - 1) * n_out + f)) = acc;
                st_acc[4 * (parts - 1) * n_out + (my_part - 1) * n_out + f] = l;
            }
            __syncthreads();
            if (my_part > 0) break;
            for (int p = 1; p < parts; ++p) {
                acc += *(MI355_LDS const float4v*)(st_acc + 4 * ((p - 1) * n_out + f));
                l += st_acc[4 * (parts - 1) * n_out + (p - 1) * n_out + f];
            }
        }
        MI355_TL(tl[6] = timeline::wall_clock();)
        store_out(f, acc, st_mc[c], l);
    }
    // ready for the next call that uses this workspace (a device-scope store like the tickets, which are the only other
    // accesses to the counter; the next launch on the stream starts after this one has ended)
    if (tid == 0) __hip_atomic_store(&counters[(long)bh * kCounterStride], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    MI355_TL(wait_vmcnt<0>(); tl[7] = timeline::wall_clock(); tl_dump();)
}

// Sets the counters of a workspace whose contents are unknown (a caller's) to zero.
__global__ void fmha_decode_clear_kernel(unsigned* counters, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) counters[i] = 0u;
}

static hipError_t clear_counters(void* counters, long n, hipStream_t stream) {
    fmha_decode_clear_kernel<<<dim3(4), dim3(256), 0, stream>>>(static_cast<unsigned*>(counters), (int)n);
    return hipGetLastError();
}

// Few query rows per kv head: this kernel, except over a short cache where the prefill kernel is expected to be done first. It
// walks up to 32 columns of queries side by side and combines its waves column by column, which with many columns takes
// longer than a short walk over the keys; the prefill kernel pads every head's queries to 128 rows, but has a workgroup per
// query head, and pays only from 256 of those on. us from the operators, operands from HBM, prefill kernel / this one: 1 x 32/8 heads, 8 queries over
// 300 keys 9.3 / 11; 8 x 32/32, 17 queries over 128 9.0 / 9.6; 16 x 32/1, 1 over 100 12.5 / 8.4; 16 x 32/8, 8 over 65 12.7 / 8.8; 8 x 64/8,
// 4 over 128 12.3 / 8.7; 20 x 32/32, 12 over 8 14.1 / 8.3; 64 x 32/32, 12 over 33 34.7 / 20.0. Over 420 calls of 17 .. 32 columns (2 .. 512 workgroups,
// 40 .. 511 keys) the model takes .6 % longer than the faster kernel on average, 1.36 times at worst (8 x 32/32, 20 over 256 16.3 / 12.0); over 80
// of up to 16 columns over up to 64 keys .2 % and 1.35 times. The constants of the kernel's 32-column instructions that it had before took 2.4 % and
// 5.2 % longer; up to 16 columns over more keys: 2 x 16/4, 4 queries over 112 keys 7.4 / 6.1, 1 x 32/8, 4 over 300 9.3 / 7.1.
bool fmha_decode_applicable(int B, int Hq, int Hkv, int Sq, int Sk, int kv_valid_len) {
    const long cols = (long)(Hq / Hkv) * Sq;
    if (cols > 32 || Sk < kv_valid_len || B < 1) return false;
    if (kv_valid_len >= 512) return true;
    const float tiles64 = (float)((kv_valid_len + 63) / 64), tiles32 = (float)((kv_valid_len + 31) / 32);
    const long items = (long)B * Hq, wgs = (long)B * Hkv;
    const float prefill_us = 4.9f + .78f * tiles64 + (float)((items + 255) / 256 - 1) * (2.4f + 1.09f * tiles64);
    const float step_us = kv_valid_len <= 64 && wgs > 256   // two waves, two workgroups to a CU
                              ? (float)((wgs + 511) / 512) * (3.5f + .11f * (float)cols + .033f * (float)kv_valid_len)
                          : cols > 16
                              ? (float)((wgs + 255) / 256) * (4.2f + .1f * (float)cols + 1.05f * ceilf(tiles32 / 4.f))
                          : kv_valid_len > 64
                              ? (float)((wgs + 255) / 256) * (3.f + .13f * (float)cols + .6f * ceilf(tiles32 / 4.f))
                              : (float)((wgs + 255) / 256) * (3.5f + .225f * (float)cols + 1.1f);
    return step_us <= 1.03f * prefill_us;
}

constexpr size_t kStaticScratchBytes = size_t(4) << 20;   // see `scratch` below
namespace dec {
constexpr int kMaxSplits = 256;   // key ranges per (batch, kv head)
}

// How a call is cut into workgroups, and what its workspace holds: one counter per (batch, kv head), kCounterStride
// words apart, then the partial results [workgroup][column][PART_STRIDE].
struct DecodePlan {
    int splits, tiles_per_split;
    int waves;                     // of a workgroup
    long workgroups;
    size_t counter_bytes, bytes;   // bytes == 0: a single key range per (batch, kv head), no workspace
    size_t ask_bytes;              // what a caller is asked for: as much as any cut the model may choose would take
};
// The most key ranges the model may choose: at least two tiles each, at most 512 workgroups, the partial results within the
// static array.
static long finer_splits(long pairs, int tiles, int ncols) {
    using namespace dec;
    const long fit = (long)((kStaticScratchBytes - kCounterBytes) / (PART_STRIDE * sizeof(float))) / (pairs * ncols);
    return std::min({(long)(tiles + 1) / 2, (long)kMaxSplits, 512 / pairs, fit});
}

static DecodePlan decode_plan(int B, int Hq, int Hkv, int Sq, int kv_valid) {
    using namespace dec;
    const int ncols = (Hq / Hkv) * Sq;
    const int tiles = (kv_valid + TK - 1) / TK;
    const long pairs = (long)B * Hkv;
    // The number of key ranges. At least about one workgroup per CU of at least eight tiles each, and more of them where that
    // is expected to be done first; never fewer, although fewer would often be faster where that many workgroups start a second
    // round for a few of them. A wave rounds its probabilities against the maximum of its first tile: the largest ones,
    // which carry most of the error, are exact there, and a longer piece more often holds larger ones behind that tile
    // (relative error of O against float64 with a half or a third of the ranges: 1.01 .. 1.05 times as large; with two to
    // four times as many 0.91 .. 1.00). The model: a workgroup (one to a CU) takes ~3 us and, per tile, what it gets of the
    // memory's rate: 0.32 us while up to 64 of them run, 0.38 with 128, 0.69 with all 256 (measured over 8192 keys); then
    // the merge. Below 512 keys one workgroup walks them all: no workspace is needed, and the merge would take as long as
    // the walk. us, with the even cut / by this rule: 8 pairs over 1000 keys 9.1 / 8.0, 52 pairs over 8191 keys (five ranges are
    // 260 workgroups) 56.8 / 45.9, 160 pairs over 4500 keys 82.8 / 70.0. (The 3 us and the merge are those of an earlier combine and
    // merge; over 84 drawn calls, 512 .. 30000 keys from HBM, the number that they give takes .8 % longer than the best of those allowed on
    // average, at worst 5 %: 16 pairs over 1704 keys 7 ranges 10.1, 16 ranges 9.6.)
    long splits = 1, most = 1;
    if (pairs <= kMaxSplitPairs && kv_valid >= 512) {
        const long even = std::max(1L, std::min({(256 + pairs / 2) / pairs, (long)(tiles + 7) / 8, (long)kMaxSplits}));
        const long even_tiles = (tiles + even - 1) / even;
        splits = (tiles + even_tiles - 1) / even_tiles;
        const auto split_us = [&](long s) {
            const float range_tiles = (float)(((tiles + s - 1) / s + 3) / 4 * 4);   // the four waves walk equal pieces
            const long full = pairs * s / 256, rest = pairs * s % 256;
            const auto round_us = [&](long wgs) {
                return 3.f + range_tiles * (wgs <= 64 ? .32f : wgs <= 128 ? .32f + .001f * (float)(wgs - 64) : .38f + .00242f * (float)(wgs - 128));
            };
            return (float)full * round_us(256) + (rest > 0 ? round_us(rest) : 0.f) + 2.5f + .04f * (float)s + (s > 24 ? .03f * (float)(s - 24) : 0.f);
        };
        // More only where the partial results fit the static array (and with it the smallest buffer of a stream): such a call
        // needs no more memory than it would with the even cut.
        most = splits > 1 ? std::max(splits, finer_splits(pairs, tiles, ncols)) : 1;
        float best_us = most > splits ? .97f * split_us(splits) : 0.f;   // (a predicted gain of less than 3 % is none)
        for (long s = splits + 1; s <= most; ++s) {
            const float us = split_us(s);
            if (us < best_us) {
                best_us = us;
                splits = s;
            }
        }
    }
    DecodePlan p;
    p.tiles_per_split = (int)((tiles + splits - 1) / splits);
    p.splits = (tiles + p.tiles_per_split - 1) / p.tiles_per_split;
    p.workgroups = pairs * p.splits;
    // Two tiles or fewer and more workgroups than CUs: two waves and 64 KiB per workgroup, so that two share a CU and one's
    // start-up and combine hide under the other's keys (us, four / two waves, 64 keys: 512 workgroups of 4 columns 10.4 / 7.5, 1024
    // workgroups 20.3 / 14.3). Each wave has one tile either way; beyond that, longer pieces would round coarser (see above).
    p.waves = kv_valid <= 2 * TK && p.workgroups > 256 ? 2 : 4;
    const auto bytes_of = [&](long s) { return s > 1 ? kCounterBytes + (size_t)(pairs * s) * ncols * PART_STRIDE * sizeof(float) : 0; };
    p.counter_bytes = p.splits > 1 ? kCounterBytes : 0;
    p.bytes = bytes_of(p.splits);
    // The number the model chooses goes up and down as the cache grows; the most it may choose only goes up (and the even cut
    // by less than a tenth down, where its last range is a short one). A caller who asks once, for the longest cache, has
    // enough for the shorter ones.
    p.ask_bytes = bytes_of(most);
    return p;
}

void fmha_decode_plan_of(int B, int Hq, int Hkv, int Sq, int kv_valid_len, int* splits, int* waves) {
    const DecodePlan plan = decode_plan(B, Hq, Hkv, Sq, kv_valid_len);
    *splits = fmha_decode_applicable(B, Hq, Hkv, Sq, kv_valid_len, kv_valid_len) ? plan.splits : 0;
    *waves = plan.waves;
}

size_t fmha_decode_workspace_bytes(int B, int Hq, int Hkv, int Sq, int Sk, int kv_valid_len) {
    if (!fmha_decode_applicable(B, Hq, Hkv, Sq, Sk, kv_valid_len)) return 0;
    return decode_plan(B, Hq, Hkv, Sq, kv_valid_len).ask_bytes;
}

// The library's own workspace: one buffer per (device, stream), allocated on first use and replaced by a larger one when
// a call needs more. A buffer that has been handed to a kernel is NEVER freed: a HIP graph captured earlier may hold
// its address, so replaced buffers stay allocated until the process ends (each replacement is at least 1.5x larger, so
// together they hold less than three times the largest request), and so does the buffer of every stream that ever made
// such a call (at least 4 MiB each: a process that creates streams without end should hand in its own workspace,
// mi355_fmha_fwd_ws). Calls on one stream are ordered, so they can share a buffer; calls on different streams get
// different ones. Nothing can be allocated while the stream is capturing: such a call fails with
// hipErrorStreamCaptureUnsupported unless an earlier call on the same stream already made the buffer large enough (run
// the step once before capturing it, or hand in a workspace of your own); a capture on another stream goes on undisturbed
// (workspace_malloc). The ticket
// counters of a new buffer are set to zero here, on the calling stream, in front of whatever uses it (no synchronous fill of the
// whole buffer on the null stream). `order` comes back holding the lock of that (device, stream): the caller keeps it until
// its kernel is issued, so that no call of another thread on the same stream, with a buffer that has grown meanwhile or not
// been cleared yet, comes between.
static hipError_t decode_workspace(size_t bytes, hipStream_t stream, char** out, std::unique_lock<std::mutex>* order) {
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
        const size_t want = bytes < (size_t(4) << 20) ? (size_t(4) << 20) : bytes + bytes / 2;
        void* fresh = nullptr;
        e = workspace_malloc(&fresh, want);
        if (e != hipSuccess) return e;
        b.ptr = fresh;   // the previous buffer, if any, stays allocated (see above)
        b.size = want;
        if (e = clear_counters(b.ptr, (long)(dec::kCounterBytes / sizeof(unsigned)), stream); e != hipSuccess) {
            b.size = 0;   // counters not cleared: the next call starts over
            return e;
        }
    }
    *out = static_cast<char*>(b.ptr);
    return hipSuccess;
}

// Static scratch for callers that must not allocate (mi355_fmha_fwd_noalloc): a fixed array in device memory, one copy
// per GPU the library is loaded on, held until the process ends; it starts out zeroed (so do its ticket counters). Host
// code never uses the symbol's name as an address: the device address is looked up once per device with
// hipGetSymbolAddress and kept. Every call on a GPU shares that GPU's array and relies on finding its ticket counters at
// zero, where every completed call leaves them: calls that overlap on one GPU race, and a call that does not run to its end
// (a kernel that is aborted, overlapping calls) leaves a counter that is not zero. From then on no workgroup of that
// (batch, kv head) draws the last ticket, O and LSE of its rows are not written and no error is reported, until the
// process ends; mi355_fmha_fwd_ws (counters zeroed on every call) is the entry point that does not depend on history.
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

size_t fmha_decode_static_scratch_bytes() { return kStaticScratchBytes; }

static hipError_t static_scratch_ptr(char** out) {
    constexpr int kMaxDevices = 64;
    static std::atomic<void*> ptrs[kMaxDevices] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    void* p = ptrs[dev].load(std::memory_order_acquire);
    if (p == nullptr) {   // threads may race here; every one of them gets the same address for this device
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (p == nullptr) return hipErrorInvalidSymbol;
        ptrs[dev].store(p, std::memory_order_release);
    }
    *out = static_cast<char*>(p);
    return hipSuccess;
}

template <typename T, int WAVES, int NSTAGE, int NB>
static hipError_t launch_decode(const T* Q, const T* K, const T* V, T* O, float* LSE, float* part, unsigned* counters, int B,
                                int Hq, int Hkv, int Sq, int Sk, float scale_log2, int causal, int kv_valid, int splits,
                                int tiles_per_split, long workgroups, const FmhaStrides& sd, hipStream_t stream) {
    constexpr int LDS = WAVES * NSTAGE * dec::STAGE_BYTES;
    static_assert(LDS >= WAVES * (32 * dec::D + 64) * 4 + 64, "the combine step reuses the pipeline memory");
    static_assert(WAVES < 4 || LDS >= (3 * dec::kMaxSplits * 32 + 32 + 64 + 5 * WAVES * 64) * 4, "so does the merge of the key ranges");
    auto kern = fmha_decode_kernel<T, WAVES, NSTAGE, NB>;
    static DynamicLdsOnce lds_once;
    if (hipError_t e = lds_once.ensure(reinterpret_cast<const void*>(kern), LDS); e != hipSuccess) return e;
    if (workgroups > 0x7fffffffL) return hipErrorInvalidValue;
    kern<<<dim3((unsigned)workgroups), dim3(WAVES * 64), LDS, stream>>>(Q, K, V, O, LSE, part, counters, B, Hq, Hkv, Sq, Sk, scale_log2,
                                                                         causal, kv_valid, splits, tiles_per_split, sd,
                                                                         DecodeMap{Hq / Hkv, divisor_of(splits), divisor_of(Hkv), divisor_of(Sq)});
    return hipGetLastError();
}

template <typename T>
hipError_t fmha_decode_dispatch(const T* Q, const T* K, const T* V, T* O, float* LSE, int B, int Hq,
                                int Hkv, int Sq, int Sk, float scale, int causal, int kv_valid, const FmhaStrides& sd,
                                const FmhaWorkspace& ws, hipStream_t stream) {
    using namespace dec;
    const DecodePlan plan = decode_plan(B, Hq, Hkv, Sq, kv_valid);
    char* wsp = nullptr;
    hipError_t e = hipSuccess;
    std::unique_lock<std::mutex> order;   // of the library's buffer, until the kernel below is issued
    if (plan.bytes > 0) {
        // Ticket counters must be zero when the kernel starts. The library's buffers and the static array are zeroed once
        // (a fresh buffer by decode_workspace, the static array by the loader) and every call leaves its counters at
        // zero; a caller's memory holds anything, so this call's counters are zeroed on every call.
        switch (ws.kind) {
            case FmhaWorkspace::kCaller:
                if (ws.ptr == nullptr || ws.bytes < plan.bytes || reinterpret_cast<uintptr_t>(ws.ptr) % 16 != 0) return hipErrorInvalidValue;
                wsp = static_cast<char*>(ws.ptr);
                e = clear_counters(wsp, (long)B * Hkv * kCounterStride, stream);
                break;
            case FmhaWorkspace::kStatic:
                if (plan.bytes > kStaticScratchBytes) return hipErrorOutOfMemory;   // the entry point checks first and says why
                e = static_scratch_ptr(&wsp);
                break;
            default:
                e = decode_workspace(plan.bytes, stream, &wsp, &order);
                break;
        }
        if (e != hipSuccess) return e;
    }
    float* part = reinterpret_cast<float*>(wsp + plan.counter_bytes);
    unsigned* counters = reinterpret_cast<unsigned*>(wsp);
    const float scale_log2 = scale * 1.4426950408889634f;
    const bool wide = (Hq / Hkv) * Sq > 16;   // two blocks of 16 columns
    const auto launch = plan.waves == 2 ? (wide ? &launch_decode<T, 2, 2, 2> : &launch_decode<T, 2, 2, 1>) : (wide ? &launch_decode<T, 4, 2, 2> : &launch_decode<T, 4, 2, 1>);
    return launch(Q, K, V, O, LSE, part, counters, B, Hq, Hkv, Sq, Sk, scale_log2, causal, kv_valid, plan.splits, plan.tiles_per_split,
                  plan.workgroups, sd, stream);
}

template hipError_t fmha_decode_dispatch<half_t>(const half_t*, const half_t*, const half_t*, half_t*, float*, int, int, int, int,
                                                  int, float, int, int, const FmhaStrides&, const FmhaWorkspace&, hipStream_t);
template hipError_t fmha_decode_dispatch<bf16_t>(const bf16_t*, const bf16_t*, const bf16_t*, bf16_t*, float*, int, int, int, int,
                                                 int, float, int, int, const FmhaStrides&, const FmhaWorkspace&, hipStream_t);

}  // namespace mi355

#ifdef MI355_TIMELINE
// profiling build: copies the records of the last generation-step attention launch to the host
extern "C" int mi355_timeline_read_fmha_decode(void* dst, size_t bytes) {
    const size_t all = sizeof(unsigned long long) * mi355::timeline::kMaxWorkgroups * mi355::timeline::kSlots;
    return (int)hipMemcpyFromSymbol(dst, HIP_SYMBOL(mi355::fmha_decode_stamps), bytes < all ? bytes : all);
}
#endif
