// Fused multi-head attention forward for gfx950 (MI355X), head_dim 128, fp16 in/out, fp32 softmax statistics.
//
// Replaces the reference's attention ladder (kernels/fmha/pkg/fmha_unified/csrc/{auto,semi}/fmha_*.{cu,cpp});
// semantics follow semi/fmha_2_amd.cpp: BHSD layout (:33-45), kv head = q head / (Hq/Hkv), causal rule
// "masked iff q_pos < k_pos" (:187-190), keys at or beyond the valid length masked (:191, with the off-by-one
// of the reference corrected), scale 1/sqrt(d) supplied by the caller (:320).
//
// One kernel family, fmha_fwd_pingpong_kernel<T, QB> (8 phase-locked waves per workgroup, MFMA 16x16x32; 256 or 128 queries
// per workgroup), described at its definition. Everything stays in registers between the two matrix products:
//   S^T = K * Q^T      A operand = K fragment read from LDS (ds_read_b128), B operand = Q fragment held in registers for the
//                      whole kernel. A lane then owns ONE query column per 16-query block and 4 of the 16 keys of a key
//                      block, so the softmax statistics m, l and the rescale factor are per-lane scalars.
//   P^T                exp2((S - m) * scale*log2e) in fp32, rounded to fp16; the accumulator layout of S^T is (up to a
//                      fixed permutation of the keys) the B-operand layout of the second product, so P never leaves the
//                      registers.
//   O^T += V^T * P^T   A operand = V^T fragment, read from the row-major V tile in LDS with the transposing
//                      ds_read_b64_tr_b16 in that same key order.
// K and V tiles (64 keys x 128 d) are copied global -> LDS with 16-byte direct-to-LDS copies into a ring of four slots
// per operand, 16-byte chunks XOR-swizzled so that both the b128 reads (K) and the transposing reads (V) are conflict free.
#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>
#include "fmha_items.h"
#include "mi355_common.h"
#include "mi355_serving_internal.h"
#include "mi355_timeline.h"

namespace mi355 {

// profiling build: per workgroup [wall: entry, loop start, loop end, exit; cycles: loop start, loop end; key tiles; 0]
MI355_TL(static __device__ unsigned long long fmha_fwd_stamps[timeline::kMaxWorkgroups * timeline::kSlots];)

namespace fmha {

constexpr int D = 128;            // head dim
constexpr int BN = 64;            // keys per tile
constexpr int ROW_BYTES = D * 2;  // 256
constexpr int TILE_BYTES = BN * ROW_BYTES;  // 16 KiB
constexpr float kLazyLog2 = 8.f;  // rescale only when a row maximum grows by more than 2^8

__device__ __forceinline__ int swz_k(int row) { return row & 15; }
__device__ __forceinline__ int swz_v16(int row) { return (row & 7) << 1; }   // 8 key rows x 32 bytes on distinct bank groups

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// maximum / sum over the four lanes that share l % 16
__device__ __forceinline__ float quad_max(float x) {
    x = fmaxf(x, __shfl_xor(x, 16, 64));
    return fmaxf(x, __shfl_xor(x, 32, 64));
}
__device__ __forceinline__ float quad_sum(float x) {
    x += __shfl_xor(x, 16, 64);
    return x + __shfl_xor(x, 32, 64);
}
// max(a, b, c) as one instruction. fmaxf() makes the compiler quiet possible signalling NaNs first (one extra
// v_max_f32 x, x per input); scores are never NaN here, and v_max3_f32 returns the non-NaN operands anyway.
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
// Register (index into the AHEAD fragment registers) of the i-th fragment of a matrix phase when fragments are read in
// order and consumed pairwise swapped (1, 0, 3, 2, ..): fragment i >= AHEAD goes where the fragment consumed just before its
// read was, i.e. where fragment (i - AHEAD) ^ 1 lived.
__device__ __forceinline__ constexpr int frag_reg(int i, int ahead) { return i < ahead ? i : frag_reg((i - ahead) ^ 1, ahead); }
// the same, kept in program order relative to its like
__device__ __forceinline__ float max3v(float a, float b, float c) {
    float r;
    asm volatile("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

}  // namespace fmha

// How the items of a launch are dealt out (see fmha_work_item)
struct ItemMap {
    int group, Hkv, per_rank, groups_per_xcd, xcd_shift, wgs;   // wgs: workgroups per XCD; xcd_shift 0: the launch is not cut by XCD
    Divisor by_group, by_hkv, by_rank, by_segments;
};
static ItemMap item_map(int B, int Hq, int Hkv, int segments, long blocks) {
    ItemMap m;
    const long kv_groups = (long)Hkv * B * segments;
    m.group = Hq / Hkv;
    m.Hkv = Hkv;
    m.xcd_shift = kv_groups % 8 == 0 && blocks % 8 == 0 ? 3 : 0;
    m.wgs = (int)(blocks >> m.xcd_shift);
    m.groups_per_xcd = (int)(kv_groups >> m.xcd_shift);
    m.per_rank = m.groups_per_xcd * m.group;
    m.by_group = divisor_of(m.group);
    m.by_hkv = divisor_of(Hkv);
    m.by_rank = divisor_of(m.per_rank);
    m.by_segments = divisor_of(segments);
    return m;
}

// Work item `round` of workgroup `wg`: a (batch, q head, q tile), or false when the workgroup has none left.
// A launch has at most one workgroup per CU; each walks its own list of items (no global counter: nothing to reset, nothing
// two launches could share). Workgroups with ids congruent mod 8 share an XCD (and its L2): when the (batch, kv head)
// groups divide evenly every XCD gets whole groups, so K and V are fetched from HBM once. On an XCD the items are ranked
// with the q tiles that see the most keys (causal) first and dealt out in rounds that run forwards and backwards in turn:
// the workgroup that got the heaviest item of one round gets the lightest of the next.
__device__ __forceinline__ bool fmha_work_item(int wg, int round, int q_tiles, const ItemMap& m, int& b, int& hkv, int& hq, int& q_tile) {
    const int x = wg & ((1 << m.xcd_shift) - 1), wl = wg >> m.xcd_shift;   // XCD, workgroup index on it
    const int u = round * m.wgs + ((round & 1) ? m.wgs - 1 - wl : wl);
    if (u >= m.per_rank * q_tiles) return false;
    const int rank = divide(u, m.by_rank), rem = u - rank * m.per_rank;   // per_rank: items of one q tile on this XCD
    const int gl = divide(rem, m.by_group), hin = rem - gl * m.group;
    q_tile = q_tiles - 1 - rank;
    const int kvg = x * m.groups_per_xcd + gl;
    b = divide(kvg, m.by_hkv);
    hkv = kvg - b * m.Hkv;
    hq = hkv * m.group + hin;
    return true;
}

// ---------------------------------------------------------------------------------------------------------
// Ping-pong kernel: 8 waves x 16 QB queries per workgroup, two waves per SIMD that alternate roles. A wave alternates between
//     a matrix phase : S(j+1) = K(j+1) Q^T and O += V(j)^T P(j)      (matrix pipe + LDS reads)
//     a softmax phase: S(j+1) -> P(j+1)                               (VALU; the tile copies ride along)
// separated by workgroup barriers. Waves 4..7 run one phase behind waves 0..3, so on every SIMD one wave is in its matrix
// phase while the other is in its softmax phase: the matrix pipe and the VALU are busy at the same time without relying on
// the instruction scheduler to interleave them inside one wave. The phases of the workgroup are numbered P0, P1, ...; waves
// 0..3 run the matrix phase in the even ones, waves 4..7 in the odd ones.
//
// Every product is made of MFMA 16x16x32 blocks: under the board's power limit that instruction sustains a ~14 % higher
// rate than 32x32x16 on random data. Per wave and key tile (64 keys), QB = 2:
//   S^T[kb][qb] (16 keys x 16 queries) = K[kb] Q[qb]^T      4 key blocks x 2 query blocks x 4 steps of 32 d = 32 MFMAs
//   O^T[db][qb] (16 d x 16 queries)   += V[j]^T[db] P[j][qb]^T   8 d blocks x 2 query blocks x 2 steps of 32 keys = 32 MFMAs
//   l[qb]                             += 1 P[j][qb]^T            the softmax row sums, as a ninth all-ones "d block"  = 4 MFMAs
// Lane l = 16 g + c holds, of S^T[kb][qb], keys 16 kb + 4 g + 0..3 of query 16 qb + c. The B operand of the second
// product wants 8 keys of one query per lane: the four values of block 2j and the four of block 2j + 1 are taken as they
// lie, i.e. contraction index 8 g + i of step j stands for key 32 j + 4 g + i (i < 4) or 32 j + 16 + 4 g + (i - 4); the
// V^T fragment is gathered in that same order by two transposing LDS reads (key rows 32 j + 4 g .. and 32 j + 16 + 4 g ..),
// so P never leaves the registers. The softmax statistics of a query live in the 4 lanes c, c + 16, c + 32, c + 48; they
// only talk to each other when the running reference has to move (lazy rescaling, below), which after the first tile is
// rare: the common path has no cross-lane operation at all.
//
// A wave issues about one instruction per 5 cycles when it has its SIMD to itself and one per 10-12 next to the partner
// wave's MFMAs, whatever the instruction is (scalar bookkeeping included): the phases are bound by their instruction
// COUNT, and the loop is built to need few:
//   * The K / V tiles live in a ring of NBUF = 4 slots per operand and the main loop is unrolled four times, so every LDS
//     address of a fragment read is a loop-invariant register plus an immediate offset (no address arithmetic in the
//     matrix phase), and the LDS destination of a copy is an immediate added into M0.
//   * A tile pair {K(q), V(q-1)} (read in the phases P(2q) and P(2q+1)) is copied by every wave during its softmax phase
//     three tile steps earlier, one copy instruction between two blocks of VALU work (issued together right behind a
//     barrier, the 32 copy instructions of a pair queue up in the CU's memory pipeline and hold every wave at its issue for
//     ~450 cycles). In the unrolled loop all 64 rows of the tile exist, so a copy is three instructions (M0, wait state,
//     load: the tile base is a scalar pointer that advances once per tile, the lane offset a loop-invariant register); the
//     last few tiles of a workgroup run a general loop whose copies clamp the tile index and the row.
//   * The pair is published (s_waitcnt vmcnt + barrier) at the end of P(2q-2), a whole phase before its first use, so a
//     wave reads the first fragments of its next matrix phase at the end of its softmax phase, in front of the barrier, and
//     the matrix pipe starts on operands that are already in registers.
//   * The softmax keeps, per query, the threshold that makes the exponent reference move and the negated scaled reference
//     as state (recomputed only when the reference moves): the common path is max tree, one compare, fma, exp2, pack.
// QB = query blocks of 16 per wave: 2 (256 queries per workgroup) or 1 (128 queries, for shapes with too few 256-query
// workgroups to fill the machine and for short sequences; every K / V fragment then feeds one MFMA instead of two).
// ---------------------------------------------------------------------------------------------------------
// 16-byte global -> LDS copy whose LDS address is a scalar register plus a compile-time constant (added straight into M0)
template <int IMM>
__device__ __forceinline__ void copy16_global_to_lds_at(const void* uniform_base, uint32_t lane_byte_offset, uint32_t lds_wave_base) {
    asm volatile(
        "s_add_u32 m0, %2, %3\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %0, %1"
        :
        : "v"(lane_byte_offset), "s"(uniform_base), "s"(lds_wave_base), "n"(IMM)
        : "memory", "m0", "scc");
}

// kRanges, kRangesF32: the keys are cut into `segments` ranges of seg_len keys (a multiple of 64) and a work item is (batch, range, head, q
// tile): it attends to its range only (K and V start seg * seg_len rows further on, the valid length and the causal limit
// are counted from there) and writes its O, normalised over its range, and its LSE to the partial buffers
// O [segments][B][Hq][Sq][128] and LSE [segments][B][Hq][Sq]; fmha_merge_segments_kernel combines them. For a few queries
// against a long cache, where one item per (head, q tile) would leave most CUs idle behind a long walk over the keys.
// MODE: kRanges: the partial outputs are of type T; kRangesF32: they are kept in 32 bits. kFewRows: one walk over all keys, for up to 16
// queries, which are a single block of rows of the first wave and are stored as they lie: through LDS they are a chain of its own behind the
// item, and a branch in the other kernels costs those up to 2 %. us, through LDS / as they lie: 64 x 16/2 heads, 9 queries over 64 keys 17.1 /
// 15.9, 24 x 32/8, 16 over 64 13.8 / 13.1, 12 x 64/8, 16 over 128 18.2 / 17.6.
enum { kOneWalk = 0, kRanges = 1, kRangesF32 = 2, kFewRows = 3 };
constexpr int kFewRowsMax = 16;
template <typename T, int QB, int MODE = kOneWalk>
__global__ __launch_bounds__(512, 2) void fmha_fwd_pingpong_kernel(const T* __restrict__ Q, const T* __restrict__ K,
                                                               const T* __restrict__ V, T* __restrict__ O,
                                                               float* __restrict__ LSE, int B, int Hq, int Hkv, int Sq,
                                                               int Sk, float scale_log2, int causal, int kv_valid,
                                                               int q_tiles, FmhaStrides sd, int segments, int seg_len, ItemMap map) {
    using namespace fmha;
    constexpr bool SEG = MODE == kRanges || MODE == kRangesF32;
    using V8 = typename Elem<T>::v8;
    using V4 = typename Elem<T>::v4;
    constexpr int NWAVES = 8;
    constexpr int NBUF = 4;
    constexpr int WQ = 16 * QB;          // queries per wave
    constexpr int BM = NWAVES * WQ;
    constexpr int VBUF0 = NBUF * TILE_BYTES;   // LDS: NBUF K slots, then NBUF V slots; slot q % NBUF holds K(q) and V(q - 1)
    static_assert(BN * ROW_BYTES / 1024 / NWAVES == 2, "the softmax phase carries four copy slots: two of K, two of V");

    MI355_TL(unsigned long long tl_w[4] = {timeline::wall_clock(), 0, 0, 0}; unsigned long long tl_c[2] = {0, 0};)
    extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
    MI355_LDS char* smem = (MI355_LDS char*)smem_raw;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int late = wave >> 2;  // 0: waves 0..3 (matrix phase in even phases), 1: waves 4..7 (one phase behind)
    const int g = lane >> 4;
    const int c16 = lane & 15;

    // ---- work items -------------------------------------------------------------------------------------------------
    struct Item {
        const T *Qh, *Kh, *Vh;
        T* Oh;
        int lse_row;             // (batch, q head), of a range too: row of LSE / Sq
        int q_block0;            // first query
        int kv_valid, shift;     // valid keys; key j is visible to query i iff j <= i + shift (causal)
        int n_tiles;             // key tiles; may be <= 0: no visible key for the whole work item
        int exists;              // 0: no such item, nothing else is set
    };
    const long o_row = SEG ? (long)D : sd.o_row;
    auto item_of = [&](int round) -> Item {
        // (opaque copies: the compiler would form products of these once and keep them in registers through the loop over the keys, which
        // has none to spare)
        int q_tiles_ = q_tiles;
        ItemMap map_ = map;
        asm volatile("" : "+s"(q_tiles_), "+s"(map_.per_rank), "+s"(map_.group), "+s"(map_.Hkv));
        Item it;
        int b, hkv, hq, q_tile;
        it.n_tiles = 0;
        it.exists = fmha_work_item(blockIdx.x, round, q_tiles_, map_, b, hkv, hq, q_tile);
        if (!it.exists) return it;
        it.q_block0 = q_tile * BM;
        long k0 = 0;
        if constexpr (SEG) {   // b counts (batch, range) pairs
            const int pair = b;
            b = divide(pair, map_.by_segments);
            const int seg = pair - b * segments;
            k0 = (long)seg * seg_len;
            it.lse_row = (seg * B + b) * Hq + hq;
            it.Oh = O + (long)it.lse_row * Sq * (MODE == kRangesF32 ? D * (int)(sizeof(float) / sizeof(T)) : D);
            it.kv_valid = min(max(kv_valid - (int)k0, 0), seg_len);
        } else {
            it.lse_row = b * Hq + hq;
            it.Oh = O + b * sd.o_batch + hq * sd.o_head;
            it.kv_valid = kv_valid;
        }
        it.shift = Sk - Sq - (int)k0;
        it.Qh = Q + b * sd.q_batch + hq * sd.q_head;
        it.Kh = K + b * sd.k_batch + hkv * sd.k_head + k0 * sd.k_row;
        it.Vh = V + b * sd.v_batch + hkv * sd.v_head + k0 * sd.v_row;
        int k_end = it.kv_valid;
        if (causal) k_end = min(k_end, min(it.q_block0 + BM, Sq) - 1 + it.shift + 1);
        it.n_tiles = (k_end + BN - 1) / BN;
        return it;
    };
    // The items to come are worked out 64 at a time, one per lane of the last wave, while the workgroup waits for its first loads, and
    // kept in LDS (fmha_items.h: in two halves in turn): the scalar registers have no room for two items.
    constexpr int kItemWords = sizeof(Item) / 4;
    static_assert(kItemWords <= 64, "a lane each");
    __shared__ int listed[ListedItems::kHeld][kItemWords];
    const auto write_listed = [&](int round, const Item& it) { __builtin_memcpy(listed[ListedItems::entry(round)], &it, sizeof(Item)); };
    // a listed item is read in one access, word i into lane i, and its fields are taken from there (field by field each was a wait of its own:
    // 13 x 64/8 heads x 353 causal 83.9 us, so 82.8; 12 x 64/8, 16 queries over 128 keys 18.7, 18.2)
    const auto listed_words = [&](int round) { return listed[ListedItems::entry(round)][min(lane, kItemWords - 1)]; };
    const auto item_from = [&](int words) -> Item {
        int w[kItemWords];
#pragma unroll
        for (int i = 0; i < kItemWords; ++i) w[i] = __builtin_amdgcn_readlane(words, i);
        Item it;
        __builtin_memcpy(&it, w, sizeof(Item));
        return it;
    };
    // steps of an item in which the pair that is copied (tiles j + 3 of K, j + 2 of V) is made of full tiles
    auto fast_steps = [](int n_tiles, int kv_valid) { return min(min(n_tiles, kv_valid / BN) - 3, n_tiles - 1); };
    Item cur = item_of(0);   // a launch has no more workgroups than items
    int q_wave0 = cur.q_block0 + wave * WQ;

    // Q fragments (B operand of the first product): lane holds Q[16 qb + c][32 ks + 8 g .. +7]
    V8 qf[QB][4];
    auto load_q = [&](const T* Qh, int q_wave0) {
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
            const int qrow = min(q_wave0 + qb * 16 + c16, Sq - 1);
            const T* qp = Qh + qrow * sd.q_row + 8 * g;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) qf[qb][ks] = *(const V8*)(qp + ks * 32);
        }
    };

    // copy i of this wave covers tile rows 32 i + 4 wave + lane/16, 16-byte chunk position lane%16
    const int copy_row0 = wave * 4 + (lane >> 4);
    const uint32_t k_row_bytes = (uint32_t)sd.k_row * 2, v_row_bytes = (uint32_t)sd.v_row * 2;
    const long k_tile_bytes = (long)BN * sd.k_row * 2, v_tile_bytes = (long)BN * sd.v_row * 2;
    const uint32_t lds_wave = (uint32_t)(uintptr_t)smem + (uint32_t)wave * 1024u;
    uint32_t k_lane_off[2], v_lane_off[2];   // of a tile with all 64 rows
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        k_lane_off[i] = (uint32_t)(copy_row0 + 32 * i) * k_row_bytes + ((lane & 15) ^ swz_k(copy_row0)) * 16;
        v_lane_off[i] = (uint32_t)(copy_row0 + 32 * i) * v_row_bytes + ((lane & 15) ^ swz_v16(copy_row0)) * 16;
    }
    // The ring runs on from one item to the next: pair q of an item whose pair 0 lies in slot `ring` is in slot (ring + q) % NBUF, and
    // what its last pair, n_tiles, leaves free (it has no K) is K(0) of the next item: pair n_tiles + q of this item is pair q of the next.
    // General copies, each operand from the item whose pair 0 is pair `first` of the current one: the tile index is clamped to that
    // item's last tile (past the end, where no next item follows, a copy re-reads that tile into a slot nobody reads any more) and rows
    // past the last valid key onto it (masked later, but V must not feed NaNs into 0 * V).
    struct Source {
        const T* base;
        int first, last_tile, valid;
    };
    int ring = 0;
    Source src_k = {cur.Kh, 0, cur.n_tiles - 1, cur.kv_valid}, src_v = {cur.Vh, 0, cur.n_tiles - 1, cur.kv_valid};
    auto issue_k1 = [&](int q, int i) {   // half i of K(q)
        const int tile = min(q - src_k.first, src_k.last_tile);
        const int last = src_k.valid - 1 - tile * BN;
        copy16_global_to_lds((const char*)src_k.base + tile * k_tile_bytes, k_lane_off[i] - (uint32_t)max(copy_row0 + 32 * i - last, 0) * k_row_bytes,
                             smem + ((ring + q) & (NBUF - 1)) * TILE_BYTES + (i * NWAVES + wave) * 1024);
    };
    auto issue_v1 = [&](int q, int i) {   // half i of V(q - 1)
        const int tile = max(min(q - 1 - src_v.first, src_v.last_tile), 0);
        const int last = src_v.valid - 1 - tile * BN;
        copy16_global_to_lds((const char*)src_v.base + tile * v_tile_bytes, v_lane_off[i] - (uint32_t)max(copy_row0 + 32 * i - last, 0) * v_row_bytes,
                             smem + VBUF0 + ((ring + q) & (NBUF - 1)) * TILE_BYTES + (i * NWAVES + wave) * 1024);
    };
    auto issue_first_pairs = [&]() {
        for (int q = 0; q < 3; ++q) {
            issue_k1(q, 0); issue_k1(q, 1);
            if (q > 0) { issue_v1(q, 0); issue_v1(q, 1); }
        }
    };
    // copies of the unrolled loop: tile base pointers of K(j + 3) and V(j + 2), advanced once per tile step
    const char* k_next = nullptr;
    const char* v_next = nullptr;
    // fragment addresses: loop-invariant registers, the slot and the block inside the tile are immediate offsets
    //   K fragment (key block kb, d step ks): row 16 kb + c, chunk (4 ks + g) ^ (row & 15)
    //   V^T fragment (key step j, d block db), transposing read t: key row 32 j + 16 t + 4 g + c / 4, d 16 db + 4 (c % 4) .. +3
    MI355_LDS char* k_ptr[4];
    MI355_LDS char* v_ptr[8];
    {
        const int k_base = c16 * ROW_BYTES + ((g ^ c16) << 4);
        const int v_row = 4 * g + (c16 >> 2);
        const int v_base = v_row * ROW_BYTES + (((((c16 & 3) >> 1)) ^ swz_v16(v_row)) << 4) + (c16 & 1) * 8;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) k_ptr[ks] = smem + (k_base ^ (ks << 6));
#pragma unroll
        for (int db = 0; db < 8; ++db) v_ptr[db] = smem + VBUF0 + (v_base ^ (db << 5));
    }

    float4v o[8][QB];
    constexpr bool kSumOnMatrixPipe = std::is_same<T, half_t>::value;
    float4v l_acc[QB];
    V8 ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = (T)1.0f;
    asm volatile("" : "+v"(ones));   // in vector registers for good (the compiler would re-materialise it in every matrix phase)
    // per query: exponent reference of the running sums, the score above which it has to move, and -reference * scale
    float m_run[QB], m_thr[QB], neg_ms[QB];
    const float lazy_margin = kLazyLog2 / scale_log2;

    auto pin_s = [](float4v(&s)[4][QB]) {
        if constexpr (QB == 2)
            asm volatile("" : "+v"(s[0][0]), "+v"(s[0][1]), "+v"(s[1][0]), "+v"(s[1][1]), "+v"(s[2][0]), "+v"(s[2][1]), "+v"(s[3][0]), "+v"(s[3][1]));
        else
            asm volatile("" : "+v"(s[0][0]), "+v"(s[1][0]), "+v"(s[2][0]), "+v"(s[3][0]));
    };
    auto pin_p = [](V8(&pf)[2][QB]) {
        if constexpr (QB == 2) asm volatile("" : "+v"(pf[0][0]), "+v"(pf[0][1]), "+v"(pf[1][0]), "+v"(pf[1][1]));
        else asm volatile("" : "+v"(pf[0][0]), "+v"(pf[1][0]));
    };
    auto pin_o = [&]() {
        if constexpr (QB == 2) {
            asm volatile("" : "+v"(l_acc[0]), "+v"(l_acc[1]));
#pragma unroll
            for (int db = 0; db < 8; db += 4)
                asm volatile("" : "+v"(o[db][0]), "+v"(o[db][1]), "+v"(o[db + 1][0]), "+v"(o[db + 1][1]), "+v"(o[db + 2][0]), "+v"(o[db + 2][1]),
                                  "+v"(o[db + 3][0]), "+v"(o[db + 3][1]));
        } else {
            asm volatile("" : "+v"(l_acc[0]), "+v"(o[0][0]), "+v"(o[1][0]), "+v"(o[2][0]), "+v"(o[3][0]), "+v"(o[4][0]), "+v"(o[5][0]), "+v"(o[6][0]),
                              "+v"(o[7][0]));
        }
    };

    // s_barrier as inline assembly: in front of a barrier it recognises the compiler waits for every LDS read it knows of,
    // and the fragments read ahead for the next matrix phase are meant to stay in flight across this one. Nothing else
    // crosses: the reads of a matrix phase have been consumed by its MFMAs, the copies are waited for explicitly.
    auto phase_barrier = []() { asm volatile("s_barrier" ::: "memory"); };
    // At the end of an even phase the pair of the step after next must have landed (all but this wave's four newest
    // copies), so that the barrier publishes it a whole phase ahead of its first reader. The same wait at the end of an odd
    // phase finds nothing to wait for (a wave's newest four copies are all that is outstanding there), so every phase ends
    // the same way and no wave has to know which half of the workgroup it belongs to.
    auto end_phase = [&]() { wait_vmcnt<4>(); phase_barrier(); };
    constexpr int AHEAD = 6;   // fragments in flight ahead of their MFMAs
    // fragment f of the matrix phase on the pair in ring slot `slot`: f < 16 K (ks = f / 4, kb = f % 4), f >= 16 V^T
    // (j = (f - 16) / 8, db = (f - 16) % 8); SLOT >= 0: compile-time slot, the whole offset is an immediate
    auto read_frag = [&](auto slot_c, int slot, int f) -> V8 {
        constexpr int SLOT = decltype(slot_c)::value;
        const int so = (SLOT >= 0 ? SLOT : slot) * TILE_BYTES;
        if (f < 16) {
            const int ks = f >> 2, kb = f & 3;
            return Elem<T>::frag(lds_read_b128(k_ptr[ks] + (so + kb * 16 * ROW_BYTES)));
        }
        const int j = (f - 16) >> 3, db = (f - 16) & 7;
        MI355_LDS char* p = v_ptr[db] + (so + (32 * j) * ROW_BYTES);
        return Elem<T>::frag(concat(lds_read_tr16_b64(p), lds_read_tr16_b64(p + 16 * ROW_BYTES)));
    };
    auto preload = [&](auto f0c, auto slot_c, int slot, V8(&fr)[AHEAD]) {
        constexpr int F0 = decltype(f0c)::value;
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) fr[i] = read_frag(slot_c, slot, F0 + i);
    };
    // matrix phase over fragments [F0, F1): S = K Q^T (f < 16) and O += V^T P (f >= 16); fr holds the first AHEAD fragments
    auto mfma_phase = [&](auto f0c, auto f1c, auto slot_c, int slot, float4v(&s)[4][QB], const V8(&pf)[2][QB], V8(&fr)[AHEAD]) {
        constexpr int F0 = decltype(f0c)::value, F1 = decltype(f1c)::value;
        if constexpr (F0 == 0) {
#pragma unroll
            for (int kb = 0; kb < 4; ++kb)
#pragma unroll
                for (int qb = 0; qb < QB; ++qb) s[kb][qb] = float4v{0.f, 0.f, 0.f, 0.f};
        }
        // Fragments are read in the order f = F0, F0 + 1, .. and consumed in pairs, the later-read one first: LDS reads complete
        // in order, so the wait for it covers its predecessor and a pair costs one s_waitcnt instead of two. The register a
        // fragment frees takes the next fragment in read order (frag_reg).
        auto use = [&](int f) {
            const int r = frag_reg(f - F0, AHEAD);
            if (f < 16) {
                const int ks = f >> 2, kb = f & 3;
#pragma unroll
                for (int qb = 0; qb < QB; ++qb) s[kb][qb] = Elem<T>::mfma16(fr[r], qf[qb][ks], s[kb][qb]);
            } else {
                const int j = (f - 16) >> 3, db = (f - 16) & 7;
#pragma unroll
                for (int qb = 0; qb < QB; ++qb) o[db][qb] = Elem<T>::mfma16(fr[r], pf[j][qb], o[db][qb]);
                if (kSumOnMatrixPipe && db == 3) {
#pragma unroll
                    for (int qb = 0; qb < QB; ++qb) l_acc[qb] = Elem<T>::mfma16(ones, pf[j][qb], l_acc[qb]);
                }
            }
        };
        static_assert((F1 - F0) % 2 == 0 && AHEAD % 2 == 0, "fragments come in pairs");
#pragma unroll
        for (int f = F0; f < F1; f += 2) {
            __builtin_amdgcn_sched_barrier(0);
            use(f + 1);
            if (f + AHEAD < F1) fr[frag_reg(f + AHEAD - F0, AHEAD)] = read_frag(slot_c, slot, f + AHEAD);
            __builtin_amdgcn_sched_barrier(0);
            use(f);
            if (f + 1 + AHEAD < F1) fr[frag_reg(f + 1 + AHEAD - F0, AHEAD)] = read_frag(slot_c, slot, f + 1 + AHEAD);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    using I0 = std::integral_constant<int, 0>;
    using I16 = std::integral_constant<int, 16>;
    using I32 = std::integral_constant<int, 32>;
    using Dyn = std::integral_constant<int, -1>;

    // softmax of tile `tile`. CSLOT >= 0: the four copies of the pair in ring slot CSLOT ride along, full tiles from the
    // running pointers; CSLOT == -1: general copies of pair tile + 3; CSLOT == -2: the same where that is a pair of the next item, none
    // otherwise.
    auto softmax_tile = [&](float4v(&s)[4][QB], int tile, V8(&pf)[2][QB], auto cslot_c) {
        constexpr int CSLOT = decltype(cslot_c)::value;
        auto copy = [&](auto which_c) {
            constexpr int W = decltype(which_c)::value;   // 0, 1: halves of K; 2, 3: halves of V
            if constexpr (CSLOT >= 0) {
                if constexpr (W < 2) copy16_global_to_lds_at<CSLOT * TILE_BYTES + W * NWAVES * 1024>(k_next, k_lane_off[W], lds_wave);
                else copy16_global_to_lds_at<VBUF0 + CSLOT * TILE_BYTES + (W - 2) * NWAVES * 1024>(v_next, v_lane_off[W - 2], lds_wave);
            } else if (CSLOT == -1 || src_v.first > 0) {
                if constexpr (W < 2) issue_k1(tile + 3, W);
                else issue_v1(tile + 3, W - 2);
            }
        };
        const int key0 = tile * BN;
        const bool need_mask = (key0 + BN > cur.kv_valid) || (causal && (key0 + BN - 1 > q_wave0 + cur.shift));
        copy(std::integral_constant<int, 0>{});
        if (need_mask) {
#pragma unroll
            for (int qb = 0; qb < QB; ++qb) {
                const int qi = q_wave0 + qb * 16 + c16;
                const int lim = causal ? min(cur.kv_valid - 1, qi + cur.shift) : cur.kv_valid - 1;  // last visible key
#pragma unroll
                for (int kb = 0; kb < 4; ++kb)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (key0 + kb * 16 + 4 * g + e > lim) s[kb][qb][e] = -INFINITY;
            }
        }
        // Lazy rescaling: m_run is the exponent reference of the running sums of a query (identical in its four lanes), not
        // necessarily its running maximum. A lane asks for it to move when one of ITS scores exceeds m_thr = m_run +
        // 2^kLazyLog2 / scale; then (any lane of the wave asked) the four lanes of every query agree on the tile's maximum
        // and the reference is raised to the running maximum. Otherwise P = exp2((S - m_run) c) <= 2^kLazyLog2 everywhere.
        // maximum of the 16 scores a lane holds of a query: two chains of v_max3 per query, the chains of both queries
        // interleaved (written in the order they are to run: between an instruction of an assembly statement and a
        // dependent one right behind it the compiler puts a wait state, an issue slot each)
        float mx[QB], mc[QB];
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) mx[qb] = max3v(s[0][qb][0], s[0][qb][1], s[0][qb][2]);
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) mc[qb] = max3v(s[0][qb][3], s[1][qb][0], s[1][qb][1]);
#pragma unroll
        for (int kb = 1; kb < 4; ++kb) {
#pragma unroll
            for (int qb = 0; qb < QB; ++qb) mx[qb] = max3v(mx[qb], s[kb][qb][2], s[kb][qb][3]);
            if (kb < 3) {
#pragma unroll
                for (int qb = 0; qb < QB; ++qb) mc[qb] = max3v(mc[qb], s[kb + 1][qb][0], s[kb + 1][qb][1]);
            }
        }
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) mx[qb] = max3v(mx[qb], mc[qb], mc[qb]);
        // the second copy sits between the max tree and the compare that reads its result: the compiler puts wait states
        // between an assembly statement and a dependent instruction, and these instructions take their place
        __builtin_amdgcn_sched_barrier(0);
        copy(std::integral_constant<int, 1>{});
        __builtin_amdgcn_sched_barrier(0);
        bool raise = false;
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) raise = raise || (mx[qb] > m_thr[qb]);
        if (__builtin_amdgcn_ballot_w64(raise) != 0) {
#pragma unroll
            for (int qb = 0; qb < QB; ++qb) {
                const float m_new = fmaxf(m_run[qb], quad_max(mx[qb]));
                const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
                const float alpha = fast_exp2((m_run[qb] - m_use) * scale_log2);
                m_run[qb] = m_new;
                m_thr[qb] = m_new + lazy_margin;
                neg_ms[qb] = -m_use * scale_log2;
                // in place, as assembly: left to itself the compiler writes the products to other registers, and the common
                // path (no rescale) then pays for 72 register moves to meet it at the join
                l_acc[qb] *= alpha;
#pragma unroll
                for (int db = 0; db < 8; ++db) o[db][qb] *= alpha;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
#pragma unroll
            for (int kb = 0; kb < 4; ++kb)
#pragma unroll
                for (int e = 0; e < 4; ++e) s[kb][qb][e] = __builtin_fmaf(s[kb][qb][e], scale_log2, neg_ms[qb]);
        __builtin_amdgcn_sched_barrier(0);
        copy(std::integral_constant<int, 2>{});
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
            for (int qb = 0; qb < QB; ++qb)
#pragma unroll
                for (int e = 0; e < 4; ++e) s[kb][qb][e] = fast_exp2(s[kb][qb][e]);
            if (kb == 1) {
                __builtin_amdgcn_sched_barrier(0);
                copy(std::integral_constant<int, 3>{});
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
            float ps[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                V8 pk;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (!kSumOnMatrixPipe) ps[e] += s[2 * j][qb][e] + s[2 * j + 1][qb][e];
                    pk[e] = (T)s[2 * j][qb][e];
                    pk[4 + e] = (T)s[2 * j + 1][qb][e];
                }
                pf[j][qb] = pk;
            }
            if (!kSumOnMatrixPipe) l_acc[qb][0] += (ps[0] + ps[1]) + (ps[2] + ps[3]);
        }
        if constexpr (CSLOT >= 0) {
            k_next += k_tile_bytes;
            v_next += v_tile_bytes;
        }
    };

    // ---- persistent loop over the work items of this workgroup ----------------------------------------------------------
    // The first pairs of the next item ride in the last softmax phases of the current one and its Q fragments are loaded behind the last
    // use of the current ones, so that the next item starts, when O has been normalised and stored (nothing waits for the stores), on
    // operands that are there. Requested together behind the last barrier, these 144 KiB and the 64 KiB of O took the CU, whose share of
    // memory's rate is ~56 GB/s from HBM, 17200 cycles from the last barrier of an item to the first of the next (4 x 32/32 x 1001, not
    // causal; 128-query items of 13 x 64/8 x 353, causal, 8400); so they take 5500 .. 6000 (3300 .. 3700). us, before / now: 16 x 32/8 x 512 causal
    // 86 / 76, 13 x 64/8 x 353 128-query items 102 / 83, 16 x 64/8 x 200 70 / 60, 8 x 32/8 x 1000 106 / 96, 1 x 32/8 x 4844 181 / 177, not causal
    // 4 x 32/32 x 1001 74.9 / 73.1, 5 x 32/8 x 1328 160 / 152. The unrolled loop wants pair 0 in slot 0: an item that has steps for it
    // starts there, also where that means that its first pairs can only leave behind the last barrier of the item in front (a second copy
    // of the general step in front of the loop makes the 256-query instantiation spill 400 bytes a lane).
    MI355_TL(unsigned long long tl_tiles = 0, tl_end = 0, tl_between = 0;)   // cycles from an item's last barrier to the first of the next
    load_q(cur.Qh, q_wave0);
    if (cur.n_tiles > 0) issue_first_pairs();
    const bool more_items = (long)q_tiles * Hq * B * (SEG ? segments : 1) > gridDim.x;   // of the launch, than it has workgroups
    bool landed = false;   // the current item's first pairs and Q fragments have been waited for
    for (int round = 0;;) {
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
            m_run[qb] = -INFINITY;
            m_thr[qb] = -INFINITY;
            neg_ms[qb] = 0.f;
            l_acc[qb] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int db = 0; db < 8; ++db) o[db][qb] = float4v{0.f, 0.f, 0.f, 0.f};
        }
        ++round;
        bool more = false;   // this workgroup has another item
        int n_next = 0;      // its key tiles, if its first pairs are copied while the current item is worked on
        if (more_items && ListedItems::refill(round) && wave == NWAVES - 1) write_listed(round + lane, item_of(round + lane));
        if (cur.n_tiles > 0) {
            const int n_tiles = cur.n_tiles;
            if (!landed) wait_vmcnt<0>();
            wait_lgkmcnt<0>();
            phase_barrier();
            if (late) phase_barrier();   // waves 4..7 idle during P0

            float4v s[4][QB];
            V8 pf[2][QB];
            V8 fr[AHEAD];
            MI355_TL(if (round == 1) tl_w[1] = timeline::wall_clock(); const unsigned long long tl_c0 = timeline::shader_cycles(); if (tl_end) tl_between += tl_c0 - tl_end;)
            preload(I0{}, Dyn{}, ring & (NBUF - 1), fr);
            __builtin_amdgcn_s_setprio(1);
            mfma_phase(I0{}, I16{}, Dyn{}, ring & (NBUF - 1), s, pf, fr);               // S(0) alone
            __builtin_amdgcn_s_setprio(0);
            pin_s(s);
            phase_barrier();   // (pairs 1 and 2 are there: nothing to wait for)
            // tile step j: softmax(j) (with the copies of pair j + 3), then S(j+1) and O += V(j)^T P(j) on pair j + 1
            auto step = [&](auto u_c, int j) {
                constexpr int U = decltype(u_c)::value;   // (ring + j) % NBUF in the unrolled loop, -1 in the general one
                using CopySlot = std::integral_constant<int, (U >= 0 ? (U + 3) % NBUF : -1)>;
                using ReadSlot = std::integral_constant<int, (U >= 0 ? (U + 1) % NBUF : -1)>;
                softmax_tile(s, j, pf, CopySlot{});
                pin_p(pf);
                preload(I0{}, ReadSlot{}, (ring + j + 1) & (NBUF - 1), fr);
                end_phase();
                __builtin_amdgcn_s_setprio(1);
                mfma_phase(I0{}, I32{}, ReadSlot{}, (ring + j + 1) & (NBUF - 1), s, pf, fr);
                __builtin_amdgcn_s_setprio(0);
                pin_s(s);
                pin_o();
                end_phase();
            };
            // unrolled loop: while the pair copied in step j (tiles j + 3 and j + 2) is made of full tiles
            const int j_fast = (ring & (NBUF - 1)) == 0 ? max(0, fast_steps(n_tiles, cur.kv_valid)) & ~(NBUF - 1) : 0;
            int j = 0;
            k_next = (const char*)cur.Kh + 3 * k_tile_bytes;
            v_next = (const char*)cur.Vh + 2 * v_tile_bytes;
            for (; j < j_fast; j += NBUF) {
                step(std::integral_constant<int, 0>{}, j);
                step(std::integral_constant<int, 1>{}, j + 1);
                step(std::integral_constant<int, 2>{}, j + 2);
                step(std::integral_constant<int, 3>{}, j + 3);
            }
            for (; j + 1 < n_tiles; ++j) {
                if (more_items && j + 3 >= n_tiles) {   // the copies go on to the next item: K with pair n_tiles, V with the one behind
                    const Item next = item_from(listed_words(round));
                    if (next.n_tiles > 0 && (((ring + n_tiles) & (NBUF - 1)) == 0 || fast_steps(next.n_tiles, next.kv_valid) < NBUF)) {
                        n_next = next.n_tiles;
                        src_k = {next.Kh, n_tiles, n_next - 1, next.kv_valid};
                        if (j + 2 == n_tiles) src_v = {next.Vh, n_tiles, n_next - 1, next.kv_valid};
                    }
                }
                step(Dyn{}, j);
            }
            if (more_items) {
                const Item next = item_from(listed_words(round));
                more = next.exists;
                if (more) load_q(next.Qh, next.q_block0 + wave * WQ);
            }
            softmax_tile(s, n_tiles - 1, pf, std::integral_constant<int, -2>{});
            if (n_tiles == 2 && n_next > 0) {   // two tiles have no step that copies pair n_tiles: K(0) of the next item
                issue_k1(2, 0);
                issue_k1(2, 1);
            }
            pin_p(pf);
            preload(I16{}, Dyn{}, (ring + n_tiles) & (NBUF - 1), fr);
            phase_barrier();
            mfma_phase(I16{}, I32{}, Dyn{}, (ring + n_tiles) & (NBUF - 1), s, pf, fr);     // O += V(last)^T P(last) alone
            phase_barrier();
            if (!late) phase_barrier();  // waves 0..3 idle while waves 4..7 finish
            // Behind this barrier no wave reads LDS any more. This wave's copies have landed, past the end of the item or of the
            // next one, and so have the next Q fragments: used here, in front of the stores of the epilogue, which the compiler would
            // otherwise wait for as well where it waits for the fragments.
            wait_vmcnt<0>();
#pragma unroll
            for (int qb = 0; qb < QB; ++qb) asm volatile("" : "+v"(qf[qb][0]), "+v"(qf[qb][1]), "+v"(qf[qb][2]), "+v"(qf[qb][3]));
            MI355_TL(tl_w[2] = timeline::wall_clock(); tl_end = timeline::shader_cycles(); tl_c[1] += tl_end - tl_c0; tl_tiles += (unsigned long long)n_tiles;)
        } else {
            wait_lgkmcnt<0>();
            phase_barrier();
            if (more_items) {
                const Item next = item_from(listed_words(round));
                more = next.exists;
                if (more) load_q(next.Qh, next.q_block0 + wave * WQ);
            }
        }

        // what the epilogue needs of the item just finished, then on to the next one
        T* const o_item = cur.Oh;
        const int q_item0 = q_wave0;
        float* const lse_item = LSE == nullptr ? nullptr : LSE + (long)cur.lse_row * Sq;
        if (more) {
            landed = n_next > 0;
            ring = landed ? ring + cur.n_tiles : 0;
            cur = item_from(listed_words(round));
            q_wave0 = cur.q_block0 + wave * WQ;
            src_k = {cur.Kh, 0, cur.n_tiles - 1, cur.kv_valid};
            src_v = {cur.Vh, 0, cur.n_tiles - 1, cur.kv_valid};
            if (cur.n_tiles > 0 && !landed) issue_first_pairs();
        }
        // ---- finalize: O / l, LSE: lane holds O[query 16 qb + c][d = 16 db + 4 g + 0..3] --------------------------------
        // 16 rows at a time go through this wave's 4 KiB of the slot in front of pair 0, which nobody reads or fills before the wave's own
        // copies of pair 3, so that a store instruction writes four whole rows (as they lie in the accumulators it would write 32 bytes
        // of each of 16 rows, four times as many lines for the CU's memory pipeline). Chunk k of row r lies at k ^ r.
        int lane_ = lane;
        asm volatile("" : "+v"(lane_));   // or the compiler keeps these addresses in vector registers through the loop over the keys
        const int r16 = lane_ & 15, r4 = lane_ >> 4;
        MI355_LDS char* const park = smem + ((ring - 1) & (NBUF - 1)) * TILE_BYTES + wave * 1024;
        auto park_row = [&](int row) -> MI355_LDS char* {   // rows 4 a .. 4 a + 3 in the wave's quarter a: halves of K, halves of V
            const int a = row >> 2;
            return park + (a >> 1) * VBUF0 + (a & 1) * (NWAVES * 1024) + (row & 3) * ROW_BYTES;
        };
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
            if (q_item0 + qb * 16 >= Sq) break;   // no such rows (a few queries are done 0.5 us sooner for it)
            const float l_tot = kSumOnMatrixPipe ? l_acc[qb][0] : quad_sum(l_acc[qb][0]);
            const float inv = (l_tot > 0.f) ? 1.f / l_tot : 0.f;
            if constexpr (MODE == kFewRows) {
                if (r16 < Sq) {
                    T* const row = o_item + r16 * o_row + 4 * r4;
#pragma unroll
                    for (int db = 0; db < 8; ++db) {
                        V4 v;
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = (T)(o[db][qb][e] * inv);
                        *(V4*)(row + db * 16) = v;
                    }
                    if (lse_item != nullptr && r4 == 0) lse_item[r16] = (l_tot > 0.f) ? (m_run[qb] * scale_log2 + __builtin_log2f(l_tot)) * 0.69314718055994531f : -INFINITY;
                }
                break;
            }
            if constexpr (MODE == kRangesF32) {   // 64 bytes of a row as they lie
                float* const row = reinterpret_cast<float*>(o_item) + (long)(q_item0 + qb * 16 + r16) * D + 4 * r4;
                if (q_item0 + qb * 16 + r16 < Sq) {
#pragma unroll
                    for (int db = 0; db < 8; ++db) *(float4v*)(row + db * 16) = o[db][qb] * inv;
                    if (r4 == 0) lse_item[q_item0 + qb * 16 + r16] = (l_tot > 0.f) ? (m_run[qb] * scale_log2 + __builtin_log2f(l_tot)) * 0.69314718055994531f : -INFINITY;
                }
                continue;
            }
            MI355_LDS char* const mine = park_row(r16);
#pragma unroll
            for (int db = 0; db < 8; ++db) {
                V4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = (T)(o[db][qb][e] * inv);
                *(MI355_LDS V4*)(mine + (((2 * db + (r4 >> 1)) ^ r16) << 4) + (r4 & 1) * 8) = v;
            }
            const int q_first = q_item0 + qb * 16;
            if (lse_item != nullptr && r4 == 0 && q_first + r16 < Sq)
                lse_item[q_first + r16] = (l_tot > 0.f) ? (m_run[qb] * scale_log2 + __builtin_log2f(l_tot)) * 0.69314718055994531f : -INFINITY;
            V8 row[4];
#pragma unroll
            for (int a = 0; a < 4; ++a) row[a] = *(MI355_LDS const V8*)(park_row(4 * a + r4) + ((r16 ^ (4 * a + r4)) << 4));
#pragma unroll
            for (int a = 0; a < 4; ++a)
                if (q_first + 4 * a + r4 < Sq) *(V8*)(o_item + (q_first + 4 * a + r4) * o_row + 8 * r16) = row[a];
        }
        if (!more) break;
    }
    MI355_TL(
        wait_vmcnt<0>();   // the stores of this wave have been accepted
        tl_w[3] = timeline::wall_clock();
        if (tid == 0 && blockIdx.x < timeline::kMaxWorkgroups) {
            unsigned long long* rec = fmha_fwd_stamps + (long)blockIdx.x * timeline::kSlots;
            rec[0] = tl_w[0]; rec[1] = tl_w[1]; rec[2] = tl_w[2]; rec[3] = tl_w[3];
            rec[4] = 0; rec[5] = tl_c[1]; rec[6] = tl_tiles; rec[7] = tl_between;
        })
}

// number of CUs of the current device (asked once per device)
static hipError_t compute_units(int& cus) {
    static std::atomic<int> cached[DynamicLdsOnce::kMaxDevices] = {};
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
    const bool tracked = dev >= 0 && dev < DynamicLdsOnce::kMaxDevices;
    if (tracked && (cus = cached[dev].load(std::memory_order_relaxed)) > 0) return hipSuccess;
    if (hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev); e != hipSuccess) return e;
    if (cus < 1) return hipErrorInvalidDevice;
    if (tracked) cached[dev].store(cus, std::memory_order_relaxed);
    return hipSuccess;
}

template <typename T, int QB, int MODE = kOneWalk>
static hipError_t launch_fmha_pingpong(const T* Q, const T* K, const T* V, T* O, float* LSE, int B, int Hq,
                                   int Hkv, int Sq, int Sk, float scale, int causal, int kv_valid, const FmhaStrides& sd,
                                   hipStream_t stream) {
    constexpr int BM = 128 * QB;
    constexpr int LDS = 8 * fmha::TILE_BYTES;
    auto kern = fmha_fwd_pingpong_kernel<T, QB, MODE>;
    static DynamicLdsOnce lds_once;
    if (hipError_t e = lds_once.ensure(reinterpret_cast<const void*>(kern), LDS); e != hipSuccess) return e;
    const int q_tiles = (Sq + BM - 1) / BM;
    const long items = (long)q_tiles * Hq * B;
    if (items > 0x7fffffffL) return hipErrorInvalidValue;
    // one workgroup per CU at most (128 KiB of LDS each: a CU holds one); a multiple of 8 when the (batch, kv head) groups
    // divide over the 8 XCDs, so that fmha_work_item can give every XCD whole groups
    int cus = 0;
    if (hipError_t e = compute_units(cus); e != hipSuccess) return e;
    long blocks = items < cus ? items : cus;
    if (((long)Hkv * B) % 8 == 0 && blocks >= 8) blocks &= ~7L;
    const float scale_log2 = scale * 1.4426950408889634f;
    kern<<<dim3((unsigned)blocks), dim3(512), LDS, stream>>>(Q, K, V, O, LSE, B, Hq, Hkv, Sq, Sk, scale_log2, causal, kv_valid,
                                                             q_tiles, sd, 1, 0, item_map(B, Hq, Hkv, 1, blocks));
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------------------
// A few queries against a long cache (a chunk of a prompt appended to earlier chunks): one work item per (head, q tile)
// would leave most CUs idle behind a walk over all keys, so the keys are cut into ranges, every (range, head, q tile) is
// a work item of the same kernel (MODE) and a second kernel merges the ranges:
//   O = sum_s w_s O_s / sum_s w_s,  w_s = exp(LSE_s - max_s LSE_s),  LSE = max_s LSE_s + log(sum_s w_s)
// (a range without a visible key has LSE_s = -inf and weight 0; a row without any visible key gets O = 0, LSE = -inf).
// The partial results live in a workspace of the library's own, one buffer per (device, stream), allocated at first use
// and replaced by a larger one when a call needs more (never freed: a captured graph may hold its address). A call that
// cannot get it (its stream is being captured and has none yet) runs the kernel without ranges instead.
// ---------------------------------------------------------------------------------------------------------------
constexpr int kMaxSegments = 8, kMaxSegmentsF32 = 16;

// 16 lanes per (batch, head, query), 8 output elements each: one pass over the partial results with 16-byte accesses, every load of a
// row issued before the first use. Bound by memory: 500 queries of 32 heads in 4 ranges, 21 MB, take 6.1 us (9.4 with a wave per row and
// 4-byte accesses).
template <typename T, typename P, int MAXS>
__global__ __launch_bounds__(256) void fmha_merge_segments_kernel(const P* __restrict__ Opart, const float* __restrict__ LSEpart,
                                                                  T* __restrict__ O, float* __restrict__ LSE, int B, int Hq, int Sq,
                                                                  int segments, FmhaStrides sd) {
    using V8 = typename Elem<T>::v8;
    typedef P P8 __attribute__((ext_vector_type(8)));
    const int part = threadIdx.x & 15;
    const long row = (long)blockIdx.x * 16 + (threadIdx.x >> 4);
    const long rows = (long)B * Hq * Sq;
    if (row >= rows) return;
    const int q = (int)(row % Sq);
    const long bh = row / Sq;
    const int h = (int)(bh % Hq), b = (int)(bh / Hq);
    float ls[MAXS];
    P8 vs[MAXS];
#pragma unroll
    for (int g = 0; g < MAXS; g += 4)   // in groups of four, a group only where it holds a range that exists
        if (g < segments)
#pragma unroll
            for (int s = g; s < g + 4; ++s) {
                const int sc = s < segments ? s : 0;
                ls[s] = LSEpart[(long)sc * rows + row];
                vs[s] = *(const P8*)(Opart + ((long)sc * rows + row) * fmha::D + 8 * part);
                if (s >= segments) ls[s] = -INFINITY;
            }
    float m = -INFINITY;
#pragma unroll
    for (int g = 0; g < MAXS; g += 4)
        if (g < segments)
#pragma unroll
            for (int s = g; s < g + 4; ++s) m = fmaxf(m, ls[s]);
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, denom = 0.f;
    if (m > -INFINITY) {
#pragma unroll
        for (int g = 0; g < MAXS; g += 4)
            if (g < segments)
#pragma unroll
                for (int s = g; s < g + 4; ++s) {
                    const float w = __expf(ls[s] - m);   // exp(-inf) = 0: a range without a visible key, or beyond `segments`
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc[e] += w * (float)vs[s][e];
                    denom += w;
                }
    }
    const float inv = denom > 0.f ? 1.f / denom : 0.f;
    V8 out;
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e] = (T)(acc[e] * inv);
    *(V8*)(O + b * sd.o_batch + h * sd.o_head + q * sd.o_row + 8 * part) = out;
    if (LSE != nullptr && part == 0) LSE[row] = denom > 0.f ? m + __logf(denom) : -INFINITY;
}

// `order` comes back holding the lock of that (device, stream), see split_k_workspace.
static hipError_t segment_workspace(size_t bytes, hipStream_t stream, char** out, std::unique_lock<std::mutex>* order) {
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
        entry = &bufs[std::make_pair(dev, stream)];
    }
    Buf& b = *entry;
    *order = std::unique_lock<std::mutex>(b.order);
    if (b.size < bytes) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        e = hipStreamIsCapturing(stream, &cap);
        if (e != hipSuccess) return e;
        if (cap != hipStreamCaptureStatusNone) return hipErrorStreamCaptureUnsupported;
        const size_t want = bytes < (size_t(8) << 20) ? (size_t(8) << 20) : bytes + bytes / 2;
        void* fresh = nullptr;
        e = workspace_malloc(&fresh, want);
        if (e != hipSuccess) return e;
        b.ptr = fresh;   // the previous buffer, if any, stays allocated (see above)
        b.size = want;
    }
    *out = static_cast<char*>(b.ptr);
    return hipSuccess;
}

// How a call cuts its keys: `segments` ranges (0: not cut) walked by work items of 128 `qb` queries.
// 128-query items: at most 128 of them; about one item per CU, at least 1024 keys per range (2048 where only two ranges
// fit), at most 8 ranges. Measured, 32/8 heads, causal, one walk / ranges (us): 64 queries over 8192 keys 90 / 25, 128 over
// 8192 92 / 28, 256 over 8192 92 / 44, 128 over 32768 343 / 75, 2 x 128 over 4096 50 / 29, 4 x 128 over 8192 94 / 79; two
// ranges of 1024 keys lose (512 over 2048: 29 / 33).
// 256-query items (every K / V fragment feeds two MFMAs) where they fill the machine with ranges of at least 2048 keys: at
// most 128 items, at least 192 (item, range) pairs, at most an eighth of the q tiles empty. Measured, 128- / 256-query
// items over ranges (us): 512 over 8192 81 / 69, 768 over 8192 105 (one walk) / 102, 1024 over 8192 127 (one walk) / 124,
// 256 over 32768 138 / 120, 512 over 32768 262 / 220, 1024 over 32768 493 (one walk) / 423, 2 x 256 over 8192 78 / 71,
// 64/8 heads 256 over 16384 139 / 120; but 256 over 8192 (8 ranges of 1024 keys) 44 / 45, 384 over 8192 65 / 67.
struct KeyRangePlan {
    int segments = 0;
    int qb = 1;
    bool f32 = false;   // partial outputs in 32 bits
    size_t bytes(long rows) const { return (size_t)segments * rows * (fmha::D * (f32 ? 4 : 2) + sizeof(float)); }
};

static KeyRangePlan long_cache_plan(int B, int Hq, int Sq, int kv_valid) {
    KeyRangePlan plan;
    if (kv_valid < 2048) return plan;
    const long q256 = (Sq + 255) / 256, items256 = q256 * Hq * B;
    if (Sq >= 256 && q256 * 256 - Sq <= Sq / 8 && items256 <= 128) {
        long s = 256 / items256;
        if (s > kMaxSegments) s = kMaxSegments;
        if (s > kv_valid / 2048) s = kv_valid / 2048;
        if (s >= 2 && items256 * s >= 192) {
            plan.segments = (int)s;
            plan.qb = 2;
            return plan;
        }
    }
    const long items = (long)((Sq + 127) / 128) * Hq * B;
    if (items > 128) return plan;
    long s = 256 / items;
    if (s > kMaxSegments) s = kMaxSegments;
    if (s > kv_valid / 1024) s = kv_valid / 1024;
    if (s == 2 && kv_valid < 4096) return plan;
    if (s >= 2) plan.segments = (int)s;
    return plan;
}

size_t fmha_key_range_workspace_bytes(int B, int Hq, int Hkv, int Sq, int Sk, int kv_valid_len) {
    if (fmha_decode_applicable(B, Hq, Hkv, Sq, Sk, kv_valid_len)) return 0;
    return long_cache_plan(B, Hq, Sq, kv_valid_len).bytes((long)B * Hq * Sq);
}

static bool being_captured(hipStream_t stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &status) == hipSuccess) return status != hipStreamCaptureStatusNone;
    (void)hipGetLastError();   // the null stream while another one is captured
    return true;
}

// Over shorter caches, and with a few items over any, the same where a small model expects it to be done sooner: a 128-query item takes
// 6 us and 0.7 us per key tile on an empty machine (1.0 with a workgroup on every CU), the second kernel 4.2 us and its bytes. At most as many (item, range)
// pairs as CUs, at least two key tiles per range, at most 16 ranges. What these calls held in 32 bits from end to end stays so: their
// partial outputs are not rounded. In the library's own workspace only (a caller's is asked for, and used, for long caches), and not in a call
// that is captured: such a graph holds no buffer of the library and may be replayed on any stream, as the header says of these sizes. us, one walk
// / ranges, causal: 1 x 32/8 heads, 58 queries over 2068 keys 28.4 / 16.4, 1 x 8/2, 36 over 2386 31.7 / 12.9, 1 x 16/4, 88 over 1561 23.4 / 15.9,
// 1 x 16/4, 229 over 1829 26.1 / 19.7, 1 x 64/8, 69 over 1500 22.5 / 19.3; but 1 x 32/8, 500 over 2000 28.6 / 33.2, 1 x 16/4, 882 over 1797 26.8 /
// 29.1, 1 x 32/8, 254 over 1425 23.0 / 22.7.
static KeyRangePlan short_cache_plan(int B, int Hq, int Sq, int kv_valid) {
    KeyRangePlan plan;
    const long rows = (long)B * Hq * Sq, items = (long)((Sq + 127) / 128) * Hq * B;
    const int tiles = (kv_valid + 63) / 64;
    if (items > 128 || tiles < 4) return plan;
    float best = .97f * .7f * (float)tiles;   // (a predicted gain of less than 3 % is none)
    for (int s = 2; s <= kMaxSegmentsF32 && s <= 256 / items && 2 * s <= tiles; ++s) {
        const int range = (tiles + s - 1) / s;
        if ((tiles + range - 1) / range != s) continue;   // the last range would be empty
        const float tile = .7f + .3f * std::max(0.f, (float)(items * s) / 128.f - 1.f);
        const float us = tile * (float)range + 4.2f + (float)s * (float)rows * 520e-6f / 3.f;
        if (us < best) {
            best = us;
            plan.segments = s;
        }
    }
    plan.f32 = plan.segments > 0;
    return plan;
}

size_t fmha_workspace_bytes(int B, int Hq, int Hkv, int Sq, int Sk, int kv_valid_len) {
    const size_t decode = fmha_decode_workspace_bytes(B, Hq, Hkv, Sq, Sk, kv_valid_len);
    return decode > 0 ? decode : fmha_key_range_workspace_bytes(B, Hq, Hkv, Sq, Sk, kv_valid_len);
}

template <typename T, int QB, int SEG>
static hipError_t launch_fmha_segmented(const T* Q, const T* K, const T* V, T* O, float* LSE, int B, int Hq, int Hkv, int Sq,
                                        int Sk, float scale, int causal, int kv_valid, const FmhaStrides& sd, int segments,
                                        char* caller_ws, hipStream_t stream) {
    using P = std::conditional_t<SEG == kRangesF32, float, T>;
    constexpr int LDS = 8 * fmha::TILE_BYTES;
    auto kern = fmha_fwd_pingpong_kernel<T, QB, SEG>;
    static DynamicLdsOnce lds_once;
    if (hipError_t e = lds_once.ensure(reinterpret_cast<const void*>(kern), LDS); e != hipSuccess) return e;
    const int seg_len = ((kv_valid + segments - 1) / segments + 63) & ~63;
    const long rows = (long)B * Hq * Sq;
    const size_t o_bytes = (size_t)segments * rows * fmha::D * sizeof(P);
    const size_t bytes = o_bytes + (size_t)segments * rows * sizeof(float);
    char* ws = caller_ws;   // memory of the caller (large enough: see fmha_fwd_dispatch), or the library's own
    std::unique_lock<std::mutex> order;   // both launches follow one another on the stream
    if (ws == nullptr)
        if (hipError_t e = segment_workspace(bytes, stream, &ws, &order); e != hipSuccess) return e;
    P* o_part = reinterpret_cast<P*>(ws);
    float* lse_part = reinterpret_cast<float*>(ws + o_bytes);
    const int q_tiles = (Sq + 128 * QB - 1) / (128 * QB);
    const long items = (long)q_tiles * Hq * B * segments;
    int cus = 0;
    if (hipError_t e = compute_units(cus); e != hipSuccess) return e;
    long blocks = items < cus ? items : cus;
    if (((long)Hkv * B * segments) % 8 == 0 && blocks >= 8) blocks &= ~7L;
    const float scale_log2 = scale * 1.4426950408889634f;
    kern<<<dim3((unsigned)blocks), dim3(512), LDS, stream>>>(Q, K, V, reinterpret_cast<T*>(o_part), lse_part, B, Hq, Hkv, Sq, Sk, scale_log2, causal, kv_valid,
                                                             q_tiles, sd, segments, seg_len, item_map(B, Hq, Hkv, segments, blocks));
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    auto merge = fmha_merge_segments_kernel<T, P, SEG == kRangesF32 ? kMaxSegmentsF32 : kMaxSegments>;
    merge<<<dim3((unsigned)((rows + 15) / 16)), dim3(256), 0, stream>>>(o_part, lse_part, O, LSE, B, Hq, Sq, segments, sd);
    return hipGetLastError();
}

// Expected time of a call on work items of 128 `qb` queries, beside what both kinds have in common: that of the workgroup with the most
// to do, as fmha_work_item deals the items out. An item takes 2.6 us and 1.2 us per key tile (256 queries, every K / V fragment feeding
// two MFMAs: 4.6 and 1.75); a last round of 128-query items up to a quarter less, the emptier it is (the clock rises; 528 .. 768 items over
// 2048 keys 94.5 .. 102.6 us, as 256-query items 99.9 .. 100.1). That weighs the queries a tile is padded by, the last round of items and, causal, the length of the
// heaviest item against the better kernel. Over 165 drawn calls (1 .. 15 sequences, 64 .. 8192 queries, 8 .. 64 heads, causal or not, and
// chunks over a cache) the choice is within 0.2 % of the faster one on average, at worst 11 % (8 x 32/32 x 619 causal 70 / 63); a rule on the number
// of 256-query items that preceded it, 1.7 %. us,
// 128- / 256-query items: 13 x 64/8 x 353 causal 83 / 99, 9 x 32/32 x 317 causal 34 / 42, 16 x 32/8 x 512 causal 85 / 76, 4 x 64/8 x 152 17.0 / 13.7,
// 3 x 16/4 x 917 36.6 / 29.1, 1 x 8/2 x 7441 228 / 183, 1 x 32/8 x 1331 44.7 / 35.6, 10 x 40/8 x 255 34.1 / 28.6, 8 x 64/8 x 638 causal 104 / 115.
static float one_walk_us(int qb, int cus, int B, int Hq, int Sq, int Sk, int causal, int kv_valid) {
    const float item = qb == 2 ? 4.6f : 2.6f, tile = qb == 2 ? 1.75f : 1.2f;
    const long bm = 128 * qb, q_tiles = (Sq + bm - 1) / bm, per_rank = (long)Hq * B, items = q_tiles * per_rank;
    const long wgs = std::min<long>(items, cus), rounds = (items + wgs - 1) / wgs;
    const auto rank_us = [&](long rank) {   // rank 0: the q tile that sees the most keys
        long keys = kv_valid;
        if (causal) keys = std::min<long>(keys, std::min((q_tiles - rank) * bm, (long)Sq) + Sk - Sq);
        return item + tile * (float)std::max(0L, (keys + 63) / 64);
    };
    if (rounds > 64) return (rank_us(0) + rank_us(q_tiles - 1)) * .5f * (float)items / (float)wgs;
    // the first, the last and the middle one, and the last one that has an item in the last round
    const long rest = items - (rounds - 1) * wgs, probes[4] = {0, wgs - 1, wgs / 2, (rounds - 1) % 2 == 0 ? rest - 1 : wgs - rest};
    const float last = qb == 2 ? 1.f : .76f + .24f * (float)rest / (float)wgs;
    float most = 0.f;
    for (const long w : probes) {
        float sum = 0.f;
        for (long r = 0; r < rounds; ++r)
            if (const long u = r * wgs + (r % 2 ? wgs - 1 - w : w); u < items) sum += rank_us(u / per_rank) * (r > 0 && r == rounds - 1 ? last : 1.f);
        most = std::max(most, sum);
    }
    return most;
}

template <typename T>
static hipError_t fmha_fwd_dispatch_t(const void* Q, const void* K, const void* V, void* O, float* LSE, int B, int Hq, int Hkv,
                                      int Sq, int Sk, float scale, int causal, int kv_valid_len, const FmhaStrides& sd,
                                      int variant, const FmhaWorkspace& ws, hipStream_t stream) {
    const T* q = static_cast<const T*>(Q);
    const T* k = static_cast<const T*>(K);
    const T* v = static_cast<const T*>(V);
    T* o = static_cast<T*>(O);
    // the kernels address a K/V tile with 32-bit byte offsets from its first row
    if (sd.k_row >= (1L << 24) || sd.v_row >= (1L << 24)) return hipErrorNotSupported;
    if (variant == 0 && fmha_decode_applicable(B, Hq, Hkv, Sq, Sk, kv_valid_len))
        return fmha_decode_dispatch<T>(q, k, v, o, LSE, B, Hq, Hkv, Sq, Sk, scale, causal, kv_valid_len, sd, ws, stream);
    // (variant 3: the ranges over long caches only; 4: those over shorter ones only)
    KeyRangePlan plan;
    if (variant == 0 || variant == 3) plan = long_cache_plan(B, Hq, Sq, kv_valid_len);
    if ((variant == 0 && plan.segments == 0) || variant == 4) plan = short_cache_plan(B, Hq, Sq, kv_valid_len);
    if (plan.f32 && variant == 0 && (ws.kind != FmhaWorkspace::kLibrary || being_captured(stream))) plan = {};
    const size_t range_bytes = plan.bytes((long)B * Hq * Sq);
    const bool caller_ws = ws.kind == FmhaWorkspace::kCaller && ws.ptr != nullptr && ws.bytes >= range_bytes &&
                           reinterpret_cast<uintptr_t>(ws.ptr) % 16 == 0;
    if (range_bytes > 0 && (ws.kind == FmhaWorkspace::kLibrary || caller_ws)) {
        char* const mem = caller_ws ? static_cast<char*>(ws.ptr) : nullptr;
        const auto launch = plan.f32 ? &launch_fmha_segmented<T, 1, kRangesF32> : plan.qb == 2 ? &launch_fmha_segmented<T, 2, kRanges> : &launch_fmha_segmented<T, 1, kRanges>;
        const hipError_t e = launch(q, k, v, o, LSE, B, Hq, Hkv, Sq, Sk, scale, causal, kv_valid_len, sd, plan.segments, mem, stream);
        // without the workspace (none yet on a stream that is being captured, or no memory) the keys are walked in one go
        if (variant >= 3 || (e != hipErrorStreamCaptureUnsupported && e != hipErrorOutOfMemory)) return e;
        (void)hipGetLastError();
    }
    if (variant >= 3) return hipErrorInvalidConfiguration;   // the test hook asked for key ranges where they do not apply
    if (variant == 0) {
        int cus = 0;
        if (hipError_t e = compute_units(cus); e != hipSuccess) return e;
        variant = one_walk_us(2, cus, B, Hq, Sq, Sk, causal, kv_valid_len) < one_walk_us(1, cus, B, Hq, Sq, Sk, causal, kv_valid_len) ? 2 : 1;
    }
    if (variant == 2) return launch_fmha_pingpong<T, 2>(q, k, v, o, LSE, B, Hq, Hkv, Sq, Sk, scale, causal, kv_valid_len, sd, stream);
    if (Sq <= kFewRowsMax) return launch_fmha_pingpong<T, 1, kFewRows>(q, k, v, o, LSE, B, Hq, Hkv, Sq, Sk, scale, causal, kv_valid_len, sd, stream);
    return launch_fmha_pingpong<T, 1>(q, k, v, o, LSE, B, Hq, Hkv, Sq, Sk, scale, causal, kv_valid_len, sd, stream);
}

hipError_t fmha_fwd_dispatch(const void* Q, const void* K, const void* V, void* O, float* LSE, int B, int Hq, int Hkv,
                             int Sq, int Sk, float scale, int causal, int kv_valid_len, const FmhaStrides& sd, int dtype,
                             int variant, const FmhaWorkspace& ws, hipStream_t stream) {
    if (dtype == MI355_DTYPE_BF16)
        return fmha_fwd_dispatch_t<bf16_t>(Q, K, V, O, LSE, B, Hq, Hkv, Sq, Sk, scale, causal, kv_valid_len, sd, variant, ws, stream);
    return fmha_fwd_dispatch_t<half_t>(Q, K, V, O, LSE, B, Hq, Hkv, Sq, Sk, scale, causal, kv_valid_len, sd, variant, ws, stream);
}

}  // namespace mi355

#ifdef MI355_TIMELINE
// profiling build: copies the records of the last attention forward launch (kMaxWorkgroups x kSlots 64-bit values) to the host
extern "C" int mi355_timeline_read_fmha_fwd(void* dst, size_t bytes) {
    const size_t all = sizeof(unsigned long long) * mi355::timeline::kMaxWorkgroups * mi355::timeline::kSlots;
    return (int)hipMemcpyFromSymbol(dst, HIP_SYMBOL(mi355::fmha_fwd_stamps), bytes < all ? bytes : all);
}
#endif
