// Paged prefill attention for gfx950.
//
// Contract (crates/swiftllm-cuda/src/bindings.rs:33-54 declares the launch;
// crates/swiftllm-core/src/memory/paged_attention.rs:154-189 lists the steps:
// scores Q K^T / sqrt(d), causal mask, softmax, times V, with K and V stored
// into the cache by slot_mapping). The reference computes none of it. Here:
//   the query tokens of the batch are packed: sequence s owns tokens
//   [start_s, start_s + L_s), start_s = sum of context_lens before s, and
//   token p of s sits in the cache at slot_mapping[start_s + p] (the caller
//   writes K/V there first, e.g. with reshape_and_cache);
//   out[start_s + i, h] = sum_{j <= i} softmax_j(scale q[start_s + i, h] .
//                         K(slot[start_s + j], kvh)) V(slot[start_s + j], kvh)
//   with kvh = h / (H / Hkv). fp16 in and out, fp32 accumulation.
// The slots of a sequence must follow its block table from position 0
// (slot of p = table[p / 16] * 16 + p % 16, what get_slot_mapping produces):
// the kernel reads the block of 16 positions from the slot of the first.
//
// Work decomposition. A wave owns two groups of 16 MFMA query rows; a group
// is tpw = 16 / gw consecutive query tokens times gw = min(G, 16) query heads
// of one kv head, and the second group takes the next tpw tokens. Every K/V
// tile the wave loads serves both groups, and the K tile is transposed once
// for both. The wave walks the key blocks up to its last token; each lane's
// query row carries its own causal limit. K tiles are copied unchanged into
// the wave's LDS by direct loads and read back already transposed
// (ds_read_b64_tr_b16), and the walk goes by pairs of blocks: one softmax
// step per 32 keys, whose PV products take the two blocks' V side by side.
// Key caches that are 8- but not 16-byte aligned take the per-block MFMA
// step shared with decode (attention_core.hpp: an identity-MFMA
// transposition of K in registers). A wave's rows are complete when
// its walk ends, so it writes its outputs directly: no combine, no barriers.
// Four waves per workgroup take consecutive token groups. Each XCD runs the
// (sequence, kv head) units of its residue mod 8 one after the other, each
// unit's workgroups latest tokens first (the longest walks start first), so
// the workgroups resident on an XCD share one unit's K/V in its L2. K/V tiles are loaded
// with ordinary (cached) loads: every query group of a sequence re-reads them.
//
// That kernel serves negative and zero scales, caches that are not 16-byte
// aligned, batches of more than 1024 prompts and batches of prompts of a few
// tokens; the usual call takes
// paged_prefill_shared_kernel (below), whose waves share their stages.

#include <algorithm>
#include <type_traits>
#include "attention_core.hpp"

namespace swiftllm {
namespace {

using namespace attn;

constexpr int kPrefillWaves = 4;

struct PrefillArgs {
    f16* out;            // [T][H][D]
    const f16* q;        // [T][H][D]
    const f16* kc;
    const f16* vc;
    const int* slots;    // [T]
    const int* ctx;      // [S] query tokens per sequence
    float scale_log2;
    int S;
    int H;
    int Hkv;
    int G;               // query heads per kv head
    int nhc;             // head chunks of 16 per kv head
    int gw;              // query heads per row group: min(G, 16)
    int tpw;             // query tokens per row group: 16 / gw (a wave has two groups)
    int groups;          // workgroups per (sequence, kv head chunk) in the grid
    long long units;     // (sequence, kv head chunk) pairs: S * Hkv * nhc
    int num_blocks;      // bound on block ids; <= 0: unbounded
    bool q16, out16;     // shared stages: q and out are 16-byte aligned
    int xcds;            // shared stages: XCDs the kv heads are dealt over, 8 or 1
};

// FOLD: scale_log2 > 0 (the usual 1/sqrt(D)), whose scale then goes into the
// softmax's exp2 argument.
typedef short s4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s4 lds_s4;

// The K^T operand of one 16-row slice J from a K tile copied unchanged into
// LDS ([d][16 tokens], 2 KiB per 64 rows). With lane l reading the 8 bytes at
// element 256 J + 4 l, ds_read_b64_tr_b16 hands lane l the elements
// K[16 J + 4 (l / 16) + i][l % 16], i = 0..3: within each 16-lane group, lane
// i receives element i % 4 of lanes i / 4, + 4, + 8, + 12 (checked on the
// GPU with an in-bounds probe). That is the transposed slice in the MFMA's
// A-operand layout, the same values the identity-MFMA transposition makes.
__device__ __forceinline__ h4 read_kT(const f16* tile, int J, int lane) {
    const s4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_s4*)(const_cast<f16*>(tile) + 256 * J + 4 * lane));
    return __builtin_bit_cast(h4, v);
}

// Zeroes the V columns of the tokens past nv0 in the low halves (the pair's
// first block) and past nv1 in the high halves (its second block); nv0 and
// nv1 are the same in every lane, so this is a scalar branch.
template <int D>
__device__ __forceinline__ void mask_v_pair(int nv0, int nv1, int kg, h8 (&vp)[D / 16]) {
    if (__builtin_amdgcn_readfirstlane(min(nv0, nv1)) < kBlockTokens) [[unlikely]] {
        const int c0 = min(max(nv0 - 4 * kg, 0), 4);
        const int c1 = min(max(nv1 - 4 * kg, 0), 4);
        const unsigned long long m0 = (c0 >= 4) ? ~0ull : ((1ull << (16 * c0)) - 1ull);
        const unsigned long long m1 = (c1 >= 4) ? ~0ull : ((1ull << (16 * c1)) - 1ull);
#pragma unroll
        for (int J = 0; J < D / 16; ++J) {
            const h4 lo = __builtin_shufflevector(vp[J], vp[J], 0, 1, 2, 3);
            const h4 hi = __builtin_shufflevector(vp[J], vp[J], 4, 5, 6, 7);
            vp[J] = cat8(mask_h4(lo, m0), mask_h4(hi, m1));
        }
    }
}

// Steps 3 + 4 for one group of 16 query rows over a pair of key blocks (32
// keys), from the S^T accumulators s0 (first block) and s1 (second): lane
// (r, kg) holds S^T[t = 4kg + i][g = r] of each. The same online softmax as
// the per-block step (lazy rescaling, weights 2^kPExpLazy * exp2(s - m) as
// fp16 hi + lo parts, FOLD as there), with one row max per 32 keys. PV runs
// on the 16x16x32 form with k = 8q + i the token 4q + i of the first block
// for i < 4 and of the second otherwise: the A operand is the lane's V
// pieces of the two blocks side by side (vp), the B operand the two blocks'
// hi parts, then their lo parts.
template <int D, bool FOLD>
__device__ __forceinline__ void softmax_pv_pair(WaveState<D>& st, f4 s0, f4 s1, bool masked,
                                                int lim0, int lim1, int kg,
                                                const h8 (&vp)[D / 16], float scale_log2) {
    constexpr int NJ = D / 16;
    float sv[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        sv[i] = FOLD ? s0[i] : s0[i] * scale_log2;
        sv[4 + i] = FOLD ? s1[i] : s1[i] * scale_log2;
    }
    if (masked) [[unlikely]] {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (4 * kg + i >= lim0) sv[i] = -INFINITY;
            if (4 * kg + i >= lim1) sv[4 + i] = -INFINITY;
        }
    }
    float bm = max3(max3(sv[0], sv[1], sv[2]), max3(sv[3], sv[4], sv[5]), max2(sv[6], sv[7]));
    bm = max_over_kg(bm);
    if constexpr (FOLD) bm *= scale_log2;
    if (__any(bm > st.m + kLazyMargin)) {
        const float m_new = fmaxf(st.m, bm);
        const float alpha = rescale(st.m, m_new);
#pragma unroll
        for (int J = 0; J < NJ; ++J) st.acc[J] *= alpha;
        st.l *= alpha;
        st.m = m_new;
    }
    // No valid token seen yet: m is -inf and so is every sv; 0 keeps the
    // weights 0.
    const float m_use = (st.m == -INFINITY) ? 0.0f : st.m;
    const float c = m_use - kPExpLazy;
    float p[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        p[i] = __builtin_amdgcn_exp2f(FOLD ? __builtin_fmaf(sv[i], scale_log2, -c) : sv[i] - c);
    }
    st.l += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    h2 hh[4], ll[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        hh[i] = __builtin_amdgcn_cvt_pkrtz(p[2 * i], p[2 * i + 1]);
        ll[i] = __builtin_amdgcn_cvt_pkrtz(sub_h2_lo(p[2 * i], hh[i]),
                                           sub_h2_hi(p[2 * i + 1], hh[i]));
    }
    const h8 ph = __builtin_bit_cast(
        h8, __builtin_shufflevector(__builtin_shufflevector(hh[0], hh[1], 0, 1, 2, 3),
                                    __builtin_shufflevector(hh[2], hh[3], 0, 1, 2, 3), 0, 1, 2,
                                    3, 4, 5, 6, 7));
    const h8 pl = __builtin_bit_cast(
        h8, __builtin_shufflevector(__builtin_shufflevector(ll[0], ll[1], 0, 1, 2, 3),
                                    __builtin_shufflevector(ll[2], ll[3], 0, 1, 2, 3), 0, 1, 2,
                                    3, 4, 5, 6, 7));
#pragma unroll
    for (int J = 0; J < NJ; ++J) st.acc[J] = mfma16x32(vp[J], ph, st.acc[J]);
#pragma unroll
    for (int J = 0; J < NJ; ++J) st.acc[J] = mfma16x32(vp[J], pl, st.acc[J]);
}

// Steps 1 + 2 of a pair of key blocks for both row groups: S^T of the first
// block (s[0] group a, s[1] group b) and of the second (s[2], s[3]), K^T read
// from the pair's two K tiles in LDS (ktiles, the second D * 16 halves after
// the first). Four independent accumulator chains.
template <int D>
__device__ __forceinline__ void qk_pair_lds(f4 (&s)[4], int lane, const f16* ktiles,
                                            const QOperand<D>& qa, const QOperand<D>& qb) {
    constexpr int NJ = D / 16;
    constexpr int kTileHalfs = D * kBlockTokens;
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = f4{0, 0, 0, 0};
#pragma unroll
    for (int J = 0; J < NJ; J += 2) {
        const h8 k0 = cat8(read_kT(ktiles, J, lane), read_kT(ktiles, J + 1, lane));
        const h8 k1 = cat8(read_kT(ktiles + kTileHalfs, J, lane),
                           read_kT(ktiles + kTileHalfs, J + 1, lane));
        const h8 qA = cat8(qa.get(J), qa.get(J + 1));
        const h8 qB = cat8(qb.get(J), qb.get(J + 1));
        s[0] = mfma16x32(k0, qA, s[0]);
        s[1] = mfma16x32(k0, qB, s[1]);
        s[2] = mfma16x32(k1, qA, s[2]);
        s[3] = mfma16x32(k1, qB, s[3]);
    }
}

// LDSK: K tiles go straight from memory into LDS (global_load_lds, 16 bytes
// a lane; the key cache is 16-byte aligned) and come back transposed by
// ds_read_b64_tr_b16; otherwise through registers and an identity-MFMA
// transposition.
template <int D, bool FOLD, bool LDSK>
__global__ __launch_bounds__(64 * kPrefillWaves) __attribute__((amdgpu_waves_per_eu(2)))
void paged_prefill_kernel(const PrefillArgs a) {
    constexpr int NJ = D / 16;
    __shared__ int s_part[kPrefillWaves];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15;
    const int kg = lane >> 4;
    // Workgroups are dealt to the 8 XCDs round-robin in launch order (x
    // fastest), so blockIdx.x % 8 names the XCD. XCD x takes the units
    // (sequence, kv head chunk) x, x + 8, x + 16, ... one after the other,
    // each unit's groups latest tokens first: the workgroups an XCD runs at
    // one time share one unit's K/V in that XCD's L2, and every XCD gets
    // the same kv heads of every sequence (equal work for any lengths when
    // the kv heads divide over the XCDs).
    const long long round =
        static_cast<long long>(blockIdx.y) + static_cast<long long>(gridDim.y) * blockIdx.z;
    const long long unit = static_cast<long long>(blockIdx.x & 7) + 8 * round;
    if (unit >= a.units) return;  // the whole workgroup: no barrier is skipped
    const int per_seq = a.Hkv * a.nhc;
    const int s = static_cast<int>(unit / per_seq);
    const int yy = static_cast<int>(unit - static_cast<long long>(s) * per_seq);
    const int kvh = yy / a.nhc;
    const int hc = yy - kvh * a.nhc;
    const int gi = a.groups - 1 - static_cast<int>(blockIdx.x >> 3);  // latest tokens first

    // start_s = sum of the lengths before s (all threads share the sum).
    int part = 0;
    for (int i = threadIdx.x; i < s; i += 64 * kPrefillWaves) part += max(a.ctx[i], 0);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) part += __shfl_xor(part, d);
    if (lane == 0) s_part[w] = part;
    __syncthreads();
    int start = 0;
#pragma unroll
    for (int i = 0; i < kPrefillWaves; ++i) start += s_part[i];
    const int L = max(a.ctx[s], 0);

    // The wave's two groups of 16 query rows: tokens tq0 .. tq0 + tpw - 1
    // (group a) and the next tpw (group b).
    const int tq0 = (gi * kPrefillWaves + w) * 2 * a.tpw;
    if (tq0 >= L) return;
    const int tq_last = min(tq0 + 2 * a.tpw, L) - 1;

    // Query row r of group k: token tq0 + k * tpw + r / gw, head h0 + r % gw.
    const int rt = r / a.gw;
    const int rh = r - rt * a.gw;
    const int g = hc * 16 + rh;
    const int h = kvh * a.G + min(g, a.G - 1);
    const int tqa = tq0 + rt;
    const int tqb = tq0 + a.tpw + rt;
    const bool ok_a = (rt < a.tpw) && (tqa < L) && (g < a.G);
    const bool ok_b = (rt < a.tpw) && (tqb < L) && (g < a.G);
    const size_t qrow_a = (static_cast<size_t>(start) + min(tqa, L - 1)) * a.H + h;
    const size_t qrow_b = (static_cast<size_t>(start) + min(tqb, L - 1)) * a.H + h;

    QOperand<D> qa, qb;
    {
        const f16* pa_ = a.q + qrow_a * D + 4 * kg;
        const f16* pb_ = a.q + qrow_b * D + 4 * kg;
#pragma unroll
        for (int J = 0; J < NJ; ++J) {
            const h4 va = *reinterpret_cast<const h4*>(pa_ + 16 * J);
            const h4 vb = *reinterpret_cast<const h4*>(pb_ + 16 * J);
            qa.v[J] = ok_a ? va : h4{0, 0, 0, 0};
            qb.v[J] = ok_b ? vb : h4{0, 0, 0, 0};
        }
    }
    h4 ident;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        ident[i] = (4 * kg + i == r) ? static_cast<f16>(1.0f) : static_cast<f16>(0.0f);
    }
    const int loff = kv_elem_offset(r, 4 * kg);
    const const_int* srow = as_const(a.slots) + start;

    WaveState<D> sa, sb;
    sa.m = sb.m = -INFINITY;
    sa.l = sb.l = 0.0f;
#pragma unroll
    for (int J = 0; J < NJ; ++J) sa.acc[J] = sb.acc[J] = f4{0, 0, 0, 0};

    // Key blocks 0 .. nkb-1, double-buffered like the decode walk: the
    // steady loop runs while at least three blocks are left (both loads of
    // an iteration are real blocks, no load depends on a condition), and the
    // last one or two are peeled off.
    const int nkb = tq_last / kBlockTokens + 1;
    auto block_at = [&](int jb) {
        return __builtin_amdgcn_readfirstlane(srow[jb * kBlockTokens]) >> kBlockShift;
    };
    auto attend = [&](int jb, int b, h4 (&k)[NJ], h4 (&v)[NJ]) {
        const int base = jb * kBlockTokens;
        const int nv = block_ok(b, a.num_blocks) ? min(kBlockTokens, L - base) : 0;
        const int lim_a = ok_a ? min(max(tqa + 1 - base, 0), nv) : 0;
        const int lim_b = ok_b ? min(max(tqb + 1 - base, 0), nv) : 0;
        attend_block_pair<D, FOLD>(sa, sb, nv, lim_a, lim_b, kg, k, v, qa, qb, ident, a.scale_log2);
    };
    if constexpr (LDSK) {
        // The walk goes by pairs of key blocks (steps of 32 keys): step t
        // covers blocks 2t and 2t + 1 (the second past nkb when nkb is odd:
        // it then contributes nothing). Per step, both K tiles go into the
        // wave's LDS and both V tiles into registers, double-buffered.
        constexpr int kTileHalfs = D * kBlockTokens;
        constexpr int kDma = kTileHalfs * 2 / (64 * 16);  // 16-byte loads per lane per tile
        // Two arrays, so the compiler can tell one step's reads from the
        // other step's loads in flight (one array made it wait for those too).
        __shared__ __align__(16) f16 s_k0[kPrefillWaves * 2 * kTileHalfs];
        __shared__ __align__(16) f16 s_k1[kPrefillWaves * 2 * kTileHalfs];
        f16* const kt0 = s_k0 + w * 2 * kTileHalfs;
        f16* const kt1 = s_k1 + w * 2 * kTileHalfs;
        const int nsteps = (nkb + 1) / 2;
        // Every LDS read of a buffer has been used by an MFMA (so it has
        // returned) before the buffer is loaded again.
        auto issue = [&](int b0, int b1, f16* dst, h8 (&vp)[NJ]) {
            const int bs0 = block_ok(b0, a.num_blocks) ? b0 : 0;
            const int bs1 = block_ok(b1, a.num_blocks) ? b1 : 0;
            const f16* k0 = a.kc + kv_tile_offset(bs0, kvh, a.Hkv, D) + 8 * lane;
            const f16* k1 = a.kc + kv_tile_offset(bs1, kvh, a.Hkv, D) + 8 * lane;
#pragma unroll
            for (int j = 0; j < kDma; ++j) {
                __builtin_amdgcn_global_load_lds(k0 + 512 * j, dst + 512 * j, 16, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < kDma; ++j) {
                __builtin_amdgcn_global_load_lds(k1 + 512 * j, dst + kTileHalfs + 512 * j, 16,
                                                 0, 0);
            }
            const f16* v0 = a.vc + kv_tile_offset(bs0, kvh, a.Hkv, D) + loff;
            const f16* v1 = a.vc + kv_tile_offset(bs1, kvh, a.Hkv, D) + loff;
#pragma unroll
            for (int J = 0; J < NJ; ++J) {
                vp[J] = cat8(load_kv<false>(v0 + kv_elem_offset(16 * J, 0)),
                             load_kv<false>(v1 + kv_elem_offset(16 * J, 0)));
            }
        };
        // Steps 3 + 4 of step t for both groups. Masks apply only where a
        // key of the step lies past the wave's first query token (the causal
        // diagonal; a partial last block and the missing second block of an
        // odd walk always do) or a block id is out of the pool: a scalar
        // test. Stale K columns (tokens >= nv) only reach the score rows of
        // those tokens, which the masks (lim <= nv) replace by -inf.
        // vw: loads issued after the pair's V loads (std::integral_constant);
        // the wait for V before PV is explicit, since the compiler's count of
        // loads into LDS mixed with loads into registers cannot be relied on.
        auto finish = [&](auto vw, int t, int b0, int b1, f4 (&sc)[4], h8 (&vp)[NJ]) {
            const int base0 = 2 * t * kBlockTokens;
            const int base1 = base0 + kBlockTokens;
            const bool ok0 = block_ok(b0, a.num_blocks);
            const bool ok1 = (2 * t + 1 < nkb) && block_ok(b1, a.num_blocks);
            const bool masked = (base0 + 2 * kBlockTokens - 1 > tq0) || !ok0 || !ok1;
            const int nv0 = ok0 ? min(kBlockTokens, L - base0) : 0;
            const int nv1 = ok1 ? min(kBlockTokens, L - base1) : 0;
            const int la0 = ok_a ? min(max(tqa + 1 - base0, 0), nv0) : 0;
            const int la1 = ok_a ? min(max(tqa + 1 - base1, 0), nv1) : 0;
            const int lb0 = ok_b ? min(max(tqb + 1 - base0, 0), nv0) : 0;
            const int lb1 = ok_b ? min(max(tqb + 1 - base1, 0), nv1) : 0;
            wait_vm<decltype(vw)::value>();
            mask_v_pair<D>(nv0, nv1, kg, vp);
            softmax_pv_pair<D, FOLD>(sa, sc[0], sc[2], masked, la0, la1, kg, vp, a.scale_log2);
            softmax_pv_pair<D, FOLD>(sb, sc[1], sc[3], masked, lb0, lb1, kg, vp, a.scale_log2);
        };
        // Block ids without scalar loads in the walk (those share their wait
        // counter with the LDS reads, and every K^T read would wait for
        // them): chunks of 64 ids (the first slots of blocks 64 c .. 64 c +
        // 63 of the walk, clamped to block nkb - 1) go into the wave's LDS by
        // direct loads, chunk c + 1 while the walk is in chunk c, and a step
        // reads the ids of its two blocks with one LDS read. A chunk is
        // loaded 64 blocks before its first read; the waits of the steps in
        // between (each at most 2 * (2 kDma + 2 NJ) loads behind) retire it.
        __shared__ __align__(16) int s_ids[kPrefillWaves][2][64];
        auto load_chunk = [&](int c) {
            const int j = min(64 * c + lane, nkb - 1);
            __builtin_amdgcn_global_load_lds(srow + j * kBlockTokens, &s_ids[w][c & 1][0], 4, 0,
                                             0);
        };
        load_chunk(0);
        load_chunk(1);
        __builtin_amdgcn_s_waitcnt(0);
        int chunk = 0;
        // Ids of step t's two blocks (steps asked for in increasing order).
        auto ids_of = [&](int t, int& b0, int& b1) {
            const int j = min(2 * t, (nkb - 1) & ~1);
            if ((j >> 6) != chunk) {
                chunk = j >> 6;
                load_chunk(chunk + 1);
            }
            const int2 v = *reinterpret_cast<const int2*>(&s_ids[w][chunk & 1][j & 63]);
            b0 = __builtin_amdgcn_readfirstlane(v.x) >> kBlockShift;
            b1 = __builtin_amdgcn_readfirstlane(v.y) >> kBlockShift;
        };
        // Loads in flight behind a step's K tiles: its V tiles, then the next
        // step's K and V tiles (when there is a next step); behind its V
        // tiles, the next step's or nothing.
        constexpr int kBehindNext = 2 * NJ + 2 * kDma + 2 * NJ;
        constexpr int kBehindLast = 2 * NJ;
        const std::integral_constant<int, 2 * kDma + 2 * NJ> v_next;
        const std::integral_constant<int, 0> v_last;
        h8 vA[NJ], vB[NJ];
        f4 sc[4];
        auto qk_then_ids = [&](const f16* kt, int t_ids, int& n0, int& n1) {
            ids_of(t_ids, n0, n1);
            qk_pair_lds<D>(sc, lane, kt, qa, qb);
        };
        int tA = 0;
        int bA0, bA1, bN0, bN1;  // step tA, step tA + 1 (clamped)
        ids_of(0, bA0, bA1);
        ids_of(1, bN0, bN1);
        issue(bA0, bA1, kt0, vA);
        int left = nsteps;
        for (; left > 2; left -= 2) {
            const int tB = tA + 1;
            const int bB0 = bN0, bB1 = bN1;
            issue(bB0, bB1, kt1, vB);
            wait_vm<kBehindNext>();
            qk_then_ids(kt0, tB + 1, bN0, bN1);
            finish(v_next, tA, bA0, bA1, sc, vA);
            tA = tB + 1;
            bA0 = bN0;
            bA1 = bN1;
            issue(bA0, bA1, kt0, vA);
            wait_vm<kBehindNext>();
            qk_then_ids(kt1, tA + 1, bN0, bN1);
            finish(v_next, tB, bB0, bB1, sc, vB);
        }
        if (left == 2) {
            const int tB = tA + 1;
            issue(bN0, bN1, kt1, vB);
            wait_vm<kBehindNext>();
            qk_pair_lds<D>(sc, lane, kt0, qa, qb);
            finish(v_next, tA, bA0, bA1, sc, vA);
            wait_vm<kBehindLast>();
            qk_pair_lds<D>(sc, lane, kt1, qa, qb);
            finish(v_last, tB, bN0, bN1, sc, vB);
        } else {
            wait_vm<kBehindLast>();
            qk_pair_lds<D>(sc, lane, kt0, qa, qb);
            finish(v_last, tA, bA0, bA1, sc, vA);
        }
        // No load may still be writing this wave's LDS when it exits.
        __builtin_amdgcn_s_waitcnt(0);
    } else {
        // The next block's id (a scalar load of its first slot) is fetched
        // one block ahead, so no load waits on it; ids past the prompt's
        // last block are clamped to it.
        h4 kA[NJ], vA[NJ], kB[NJ], vB[NJ];
        int jA = 0;
        int bA = block_at(0);
        int bNext = block_at(min(1, nkb - 1));  // block jA + 1
        load_tile<D, false>(a.kc, a.vc, a.Hkv, a.num_blocks, bA, kvh, loff, kA, vA);
        int left = nkb;
        for (; left > 2; left -= 2) {
            const int jB = jA + 1;
            const int bB = bNext;
            load_tile<D, false>(a.kc, a.vc, a.Hkv, a.num_blocks, bB, kvh, loff, kB, vB);
            bNext = block_at(jB + 1);
            attend(jA, bA, kA, vA);
            jA = jB + 1;
            bA = bNext;
            load_tile<D, false>(a.kc, a.vc, a.Hkv, a.num_blocks, bA, kvh, loff, kA, vA);
            bNext = block_at(min(jA + 1, nkb - 1));
            attend(jB, bB, kB, vB);
        }
        if (left == 2) {
            const int jB = jA + 1;
            const int bB = bNext;
            load_tile<D, false>(a.kc, a.vc, a.Hkv, a.num_blocks, bB, kvh, loff, kB, vB);
            attend(jA, bA, kA, vA);
            attend(jB, bB, kB, vB);
        } else {
            attend(jA, bA, kA, vA);
        }
    }

    auto store = [&](const WaveState<D>& st, bool ok, size_t qrow) {
        float l_run = st.l;
        l_run = sum_over_kg(l_run);
        if (!ok) return;
        const float inv = (l_run > 0.0f) ? 1.0f / l_run : 0.0f;
        f16* op = a.out + qrow * D + 4 * kg;
#pragma unroll
        for (int J = 0; J < NJ; ++J) {
            h4 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = static_cast<f16>(st.acc[J][i] * inv);
            *reinterpret_cast<h4*>(op + 16 * J) = o;
        }
    };
    store(sa, ok_a, qrow_a);
    store(sb, ok_b, qrow_b);
}

// ---------------------------------------------------------------------------
// Shared stages: the prefill kernel for positive scales and 16-byte aligned
// caches, up to kSharedMaxSeqs sequences.
//
// A workgroup's four waves take consecutive tokens of one kv head, so they
// walk the same keys: each stage of 64 keys (four blocks) goes into LDS once
// for all of them, one block per wave by direct buffer loads, two stages
// deep, one barrier a stage. A wave owns 32 query rows (32 / gw tokens x gw =
// min(G, 32) heads) on v_mfma_f32_32x32x16_f16: S^T = K Q^T leaves a lane 32
// scores of one query row, so a row's maximum and sum are in-lane up to one
// lane swap, and P goes into PV straight from those registers. V lies in the
// cache as that product's row operand already; K comes back transposed by
// ds_read_b64_tr_b16, with its rows permuted so that both operands of PV are
// contiguous. The next stage's scores are made among this stage's weights.
//
// Work list. Every workgroup of a resident grid walks a list of query tiles,
// longest walk first over all sequences, each XCD its own kv heads, so no
// slot is left with a long tile at the end and no empty workgroup is launched
// for short prompts. Outputs go through LDS as whole rows, nontemporally.
//
// Bound: MFMA, at the clock the power limit leaves. On 8 x 2048 tokens the
// matrix pipes are busy 51% of the cycles at 1.75 GHz, on 1 x 8192 58% at
// 1.65 GHz (32/8 heads x 128): 1.12 PFLOP/s with the lo half of P, where
// operands in registers alone reach 1.6. Fewer VALU instructions (the lo half
// by mixed-precision multiply-adds), other interleavings of MFMA and VALU and
// wave priorities moved it by under 3% either way. Measured on one box
// (us per call, per-wave tiles -> this kernel): 8 x 2048 545 -> 443, 1 x 8192
// 887 -> 734, 1 x 2048 82 -> 66, 24 prompts of 1-2457 tokens 241 -> 190, 64
// of 16-200 60.8 -> 41.2, 4 x 1000-3000 of 16/16 heads 217 -> 157, 8 x 2048
// of 8/8 heads x 64 101 -> 66. Of that, tiles longest first
// against sequence by sequence: 208 -> 196 (24 prompts), 190 -> 165 (16/16
// heads), 88 -> 70 (x 64); whole-row outputs 54 -> 43 (64 short prompts).
// Loading the next tile's first stages and Q during a tile's last stage
// changed nothing (459 -> 470, 55 -> 55) and is not done.
// ---------------------------------------------------------------------------
constexpr int kSharedMaxSeqs = 1024;  // sequences in the LDS tile table
constexpr long long kSharedCUs = 256;  // MI355X; any grid is correct, this one is resident at once
template <int D>
constexpr int kSharedPerCU = D == 128 ? 2 : 3;  // workgroups per CU, waves per SIMD

// Query rows (tokens x heads of a kv head) of the longest prompt up to which
// the per-wave kernel is the faster one: such a prompt is one short walk, and
// finding its tile, the stage's barriers and the pass through LDS cost more
// than they save. Measured (us per call, per-wave / shared): 1 prompt of 8/8
// heads x 64 of 31 tokens 4.5 / 5.2, 94 tokens 6.1 / 6.7, 126 7.0 / 6.7; 16 of
// up to 88 tokens 6.3 / 6.8, up to 124 7.4 / 7.0; 32/8 heads x 128, 4 of up to
// 16 tokens 6.1 / 7.0, 23 tokens 7.0 / 7.0, 31 tokens 8.1 / 7.1; 64/8 x 128, 8
// tokens 6.1 / 6.9, 11 6.8 / 6.9, 16 8.0 / 7.0. With more tiles than the grid
// holds the line is lower, and where every head has its own kv head (a row is a
// token there, and walks as many keys) it lies elsewhere for each head_dim.
// Per-wave time over shared, 65 to 1000 prompts of equal lengths / of 1 up to
// the same: 2 to 8 heads to a kv head, 64 rows 0.71-1.14 / 0.66-0.96, 96 rows
// 0.96-1.43 / 0.79-1.17; 8/8 x 64, 96 rows 0.85-0.99 / 0.73-0.84, 128 rows
// 0.94-1.21 / 0.84-0.96; 16/16 x 128, 32 rows 0.85-0.99 / 0.77-0.88, 64 rows
// 0.98-1.13 / 0.90-1.10.
constexpr long long kBriefRows = 96;
constexpr long long brief_rows_many(int G, int D) { return G > 1 ? 64 : D == 64 ? 96 : 32; }

typedef float f16x __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f16x mfma32(h8 a, h8 b, f16x c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// LDS of one stage (64 keys), in halves: four K tiles [d][16], then four V
// tiles in operand order. The second K tile of a pair sits 128 bytes off, so
// that the two tiles' rows an operand read takes together fall in different
// banks.
template <int D>
struct Stage {
    static constexpr int kTile = D * kBlockTokens;
    static constexpr int kOdd = kTile + 64;
    static constexpr int kPair = 2 * kTile + 128;
    static constexpr int kK = 2 * kPair;
    static constexpr int kV = 4 * kTile;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const f16* cache, int b, int kvh, int Hkv, int D) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<f16*>(cache + kv_tile_offset(b, kvh, Hkv, D)), 0,
                                             D * kBlockTokens * 2, kRsrcWord3);
}

// Block b's K tile into its place of a K stage, copied as it is.
template <int D>
__device__ __forceinline__ void stage_k(const PrefillArgs& a, f16* ks, int w, int b, int kvh, int lane) {
    const __amdgpu_buffer_rsrc_t rk = tile_rsrc(a.kc, b, kvh, a.Hkv, D);
    f16* const k = ks + (w >> 1) * Stage<D>::kPair + (w & 1) * Stage<D>::kOdd;
#pragma unroll
    for (int i = 0; i < D / 32; ++i) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, to_lds(k + 512 * i), 16, 16u * lane, 1024u * i, 0, 0);
    }
}

// Block b's V tile into its place of a V stage, each 32-row piece's 16-byte
// chunks in operand order: the rows' first 8 tokens, then their last 8.
template <int D>
__device__ __forceinline__ void stage_v(const PrefillArgs& a, f16* vs, int w, int b, int kvh, int lane) {
    const __amdgpu_buffer_rsrc_t rv = tile_rsrc(a.vc, b, kvh, a.Hkv, D);
    f16* const v = vs + w * Stage<D>::kTile;
    const unsigned vo = 32u * (lane & 31) + 16u * (lane >> 5);
#pragma unroll
    for (int i = 0; i < D / 32; ++i) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, to_lds(v + 512 * i), 16, vo, 1024u * i, 0, 0);
    }
}

// Zeroes tokens nv .. 15 of the wave's V tile in LDS, once its loads have
// landed: stale values there (perhaps NaN) have weight 0.
template <int D>
__device__ __forceinline__ void clean_v(f16* vs, int w, int nv, int lane) {
    const int n = min(max(nv - 8 * (lane >> 5), 0), 8);
#pragma unroll
    for (int i = 0; i < D / 32; ++i) {
        h8* const p = reinterpret_cast<h8*>(vs + w * Stage<D>::kTile + 512 * i + 8 * lane);
        h8 v = *p;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = e < n ? v[e] : static_cast<f16>(0.0f);
        *p = v;
    }
}

// S^T of a 64-key stage: sc[T] the 32 keys of pair T.
template <int D>
__device__ __forceinline__ void qk_stage(f16x (&sc)[2], const f16* kl, const h8 (&q)[D / 16]) {
    sc[0] = f16x{};
    sc[1] = f16x{};
#pragma unroll
    for (int J = 0; J < D / 16; ++J) {
#pragma unroll
        for (int T = 0; T < 2; ++T) {
            const f16* p = kl + T * Stage<D>::kPair + 256 * J;
            const s4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(const_cast<f16*>(p)));
            const s4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(const_cast<f16*>(p + 64)));
            sc[T] = mfma32(cat8(__builtin_bit_cast(h4, x), __builtin_bit_cast(h4, y)), q[J], sc[T]);
        }
    }
}

// Query tiles (per_wg tokens) and token prefix of every sequence: of up to 64
// sequences in registers, one per lane (no barrier before the first tile), of
// more in LDS.
struct TileLds {
    int tiles[kSharedMaxSeqs];
    int start[kSharedMaxSeqs];  // tokens before the sequence
};

struct TileTable {
    TileLds* lds;  // S > 64
    int S;
    int tiles;     // S <= 64: of sequence `lane`
    int start;
    int top;       // tiles of the longest sequence
    __device__ __forceinline__ int tiles_of(int s0, int lane) const {
        if (S <= 64) return tiles;
        return s0 + lane < S ? lds->tiles[s0 + lane] : 0;
    }
    __device__ __forceinline__ int start_of(int s) const {
        return __builtin_amdgcn_readfirstlane(S <= 64 ? __builtin_amdgcn_readlane(start, s) : lds->start[s]);
    }
    // (tile, sequence) pairs with a tile index >= i.
    __device__ __forceinline__ int count(int i, int lane) const {
        int n = 0;
        for (int s0 = 0; s0 < S; s0 += 64) n += max(tiles_of(s0, lane) - i, 0);
        return wave_total(n);
    }
};

__device__ __forceinline__ TileTable make_tiles(const int* ctx, int S, int per_wg, int max_tiles, TileLds* lds,
                                                int* s_part) {
    TileTable t{lds, S, 0, 0, 0};
    const int lane = threadIdx.x & 63;
    if (S <= 64) {
        const int len = lane < S ? max(ctx[lane], 0) : 0;
        t.tiles = min((len + per_wg - 1) / per_wg, max_tiles);
        t.start = wave_inclusive_scan(len) - len;
        t.top = wave_max(t.tiles);
        return t;
    }
    constexpr int kEach = kSharedMaxSeqs / (64 * kPrefillWaves);
    const int c0 = threadIdx.x * kEach;
    int len[kEach];
    int sum = 0, most = 0;
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
        len[i] = c0 + i < S ? max(ctx[c0 + i], 0) : 0;
        sum += len[i];
        most = max(most, len[i]);
    }
    most = wave_max(most);
    const int incl = wave_inclusive_scan(sum);
    const int w = threadIdx.x >> 6;
    if (lane == 63) {
        s_part[w] = incl;
        s_part[kPrefillWaves + w] = most;
    }
    __syncthreads();
    for (int i = 0; i < kPrefillWaves; ++i) most = max(most, s_part[kPrefillWaves + i]);
    t.top = min((most + per_wg - 1) / per_wg, max_tiles);
    int at = incl - sum;
    for (int i = 0; i < w; ++i) at += s_part[i];
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
        if (c0 + i < S) {
            lds->tiles[c0 + i] = min((len[i] + per_wg - 1) / per_wg, max_tiles);
            lds->start[c0 + i] = at;
            at += len[i];
        }
    }
    __syncthreads();
    return t;
}

// Entry e (below count(0)) of the list of (tile, sequence) pairs, highest tile
// index (longest walk) first, sequences in order within one index. Every wave
// works it out for itself. The search starts from the longest sequence, since
// a caller's bound may lie far above it: 900 prompts of 1-2 tokens under a bound
// of 2048, 64/8 heads x 128, took 191 us from the bound and take 96.
__device__ __forceinline__ void nth_tile(const TileTable& tt, int e, int lane, int& tile, int& seq) {
    int lo = 0, hi = tt.top, below = 0;  // count(lo) > e >= count(hi) = below
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        const int n = tt.count(mid, lane);
        if (n > e) {
            lo = mid;
        } else {
            hi = mid;
            below = n;
        }
    }
    tile = lo;
    int k = e - below;  // the k-th sequence with more than `lo` tiles
    for (int s0 = 0;; s0 += 64) {
        const bool has = tt.tiles_of(s0, lane) > lo;
        const unsigned long long mask = __ballot(has);
        const int n = __popcll(mask);
        if (k < n || s0 + 64 >= tt.S) {
            const int rank = __popcll(mask & ((1ull << lane) - 1ull));
            seq = s0 + __ffsll(static_cast<long long>(__ballot(has && rank == k))) - 1;
            return;
        }
        k -= n;
    }
}

template <int D>
__global__ __launch_bounds__(64 * kPrefillWaves) __attribute__((amdgpu_waves_per_eu(kSharedPerCU<D>)))
void paged_prefill_shared_kernel(const PrefillArgs a) {
    constexpr int NJ = D / 16;   // 16-wide k steps of QK^T
    constexpr int ND = D / 32;   // 32-row pieces of the output
    using St = Stage<D>;
    __shared__ int s_part[2 * kPrefillWaves];
    __shared__ TileLds s_tiles;
    __shared__ __align__(16) f16 s_k[2][St::kK];
    __shared__ __align__(16) f16 s_v[2][St::kV];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int per_wg = kPrefillWaves * a.tpw;
    const TileTable tt = make_tiles(a.ctx, a.S, per_wg, a.groups, &s_tiles, s_part);

    // Query row r of the wave in a tile: token tq0 + r / gw, head r % gw.
    const int r = lane & 31;
    const int h = lane >> 5;
    // K operand: lane (16-lane group g4, j) reads 4 tokens of row j / 4 of
    // its 4-row piece; ds_read_b64_tr_b16 hands lane j the piece's 4 rows of
    // one token. Groups 0 and 2 take the pair's first block, 1 and 3 its
    // second, groups 2 and 3 the upper 8 of the 16 rows. The tokens of j / 4
    // = 1 and 2 are exchanged, so the products' rows 8 a + 4 h + c hold the
    // block's tokens 8 h + 4 a + c: a lane's eight scores of a block are then
    // eight consecutive tokens, and its V operand 16 contiguous bytes.
    const int g4 = lane >> 4;
    const int j = lane & 15;
    const int swapped = ((j & 1) << 1) | ((j >> 1) & 1);
    const int koff = (g4 & 1) * St::kOdd + (8 * (g4 >> 1) + (j >> 2)) * kBlockTokens + 4 * swapped;

    // Workgroups go to the 8 XCDs round-robin, so blockIdx.x % xcds names the
    // XCD (xcds is 1 when the kv heads do not divide over them). Each XCD runs
    // every sequence's tiles of its own kv heads, so a unit's K/V is read
    // through one L2. Its workgroups take the list in rounds, every other one
    // backwards.
    const unsigned x = blockIdx.x % a.xcds;
    const unsigned l0 = blockIdx.x / a.xcds;
    const unsigned wgs = gridDim.x / a.xcds;
    const unsigned heads = a.Hkv * a.nhc / a.xcds;
    const unsigned total = static_cast<unsigned>(tt.count(0, lane)) * heads;  // below 2^31 (host)
    auto item_of = [&](unsigned round) { return round * wgs + ((round & 1) ? wgs - 1 - l0 : l0); };
    for (unsigned round = 0; item_of(round) < total; ++round) {
    if (round > 0) __syncthreads();  // the stages are free for the next tile
    const unsigned item = item_of(round);
    const unsigned e = item / heads;
    int tile, s;
    nth_tile(tt, static_cast<int>(e), lane, tile, s);
    s = __builtin_amdgcn_readfirstlane(s);
    tile = __builtin_amdgcn_readfirstlane(tile);
    const int yy = static_cast<int>(x + a.xcds * (item - e * heads));
    const int kvh = yy / a.nhc;
    const int hc = yy - kvh * a.nhc;
    const int start = tt.start_of(s);
    const int L = max(as_const(a.ctx)[s], 0);
    const int wg_last = min((tile + 1) * per_wg, L) - 1;
    const int nkb = wg_last / kBlockTokens + 1;
    const int nsteps = wg_last / 64 + 1;
    // (worked out per tile behind an empty asm, so that neither stays in a
    // register through the walk)
    int rr = r;
    asm volatile("" : "+v"(rr));
    const int rt = rr / a.gw;
    const int rh = rr - rt * a.gw;
    const int g = hc * 32 + rh;
    const int head = kvh * a.G + min(g, a.G - 1);
    const int tq0 = tile * per_wg + w * a.tpw;
    const int tq = tq0 + rt;
    const bool ok = (rt < a.tpw) && (g < a.G) && tq < L;
    const size_t qrow = (static_cast<size_t>(start) + min(tq, L - 1)) * a.H + head;
    const int lim = ok ? tq + 1 : 0;                  // keys this row sees
    const int rel = ok ? rt * a.H + head : -1;        // row among the wave's tokens
    // Blocks up to the one of the wave's last token; 0: it has no token.
    const int nvis = tq0 < L ? (min(tq0 + a.tpw, L) - 1) / kBlockTokens + 1 : 0;

    const const_int* srow = as_const(a.slots) + start;
    auto chunk_ids = [&](int c) {
        return srow[static_cast<size_t>(min(64 * c + lane, nkb - 1)) * kBlockTokens] >> kBlockShift;
    };
    int ids = chunk_ids(0);
    int ids_next = chunk_ids(1);
    // Q^T operand: lane (r, h) holds q[r][16 J + 8 h .. + 7].
    h8 q[NJ];
    {
        const f16* p = a.q + qrow * D + 8 * h;
        if (a.q16) {
#pragma unroll
            for (int J = 0; J < NJ; ++J) q[J] = *reinterpret_cast<const h8*>(p + 16 * J);
        } else {
#pragma unroll
            for (int J = 0; J < NJ; ++J) {
                q[J] = cat8(*reinterpret_cast<const h4*>(p + 16 * J), *reinterpret_cast<const h4*>(p + 16 * J + 4));
            }
        }
#pragma unroll
        for (int J = 0; J < NJ; ++J) q[J] = ok ? q[J] : h8{0, 0, 0, 0, 0, 0, 0, 0};
    }
    // Block of this wave in stage u (stages asked for in order) and, in ok4,
    // which of the stage's four blocks are in the pool.
    auto block_of = [&](int u, int& ok4) {
        if (u > 0 && (u & 15) == 0) {
            ids = ids_next;
            ids_next = chunk_ids((u >> 4) + 1);
        }
        const unsigned long long okm = __ballot(block_ok(ids, a.num_blocks));
        const int at = 4 * (u & 15);
        ok4 = static_cast<int>((okm >> at) & 15ull);
        const int b = __builtin_amdgcn_readlane(ids, at + w);
        return block_ok(b, a.num_blocks) ? b : 0;
    };

    f16x acc[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) acc[i] = f16x{};
    float m = -INFINITY, l = 0.0f;

    // Tokens of this wave's block of stage u that exist.
    auto tokens_of = [&](int u, int ok4) {
        return ((ok4 >> w) & 1) ? min(max(L - (64 * u + 16 * w), 0), kBlockTokens) : 0;
    };
    int ok_t, ok_1, ok_2 = 15;  // of stages t, t + 1 and t + 2
    int b_1 = 0, b_2 = 0;
    {
        const int b = block_of(0, ok_t);
        stage_k<D>(a, s_k[0], w, b, kvh, lane);
        stage_v<D>(a, s_v[0], w, b, kvh, lane);
        ok_1 = 15;
        if (nsteps > 1) {
            b_1 = block_of(1, ok_1);
            stage_k<D>(a, s_k[1], w, b_1, kvh, lane);
        }
        wait_vm<0>();
        const int nv = tokens_of(0, ok_t);
        if (nv < kBlockTokens) clean_v<D>(s_v[0], w, nv, lane);
    }
    __syncthreads();
    f16x sc[2];
    qk_stage<D>(sc, s_k[0] + koff, q);
    __syncthreads();
    // Stage t; kMore: another follows, and its scores are made among this one's
    // weights. kAll: the wave's rows reach into each of its four blocks. The
    // workgroup walks to its last token and a wave's rows may end before; blocks
    // past them have no weight and are left out, since 0 times a value there
    // that is not finite would be NaN. (The test in every stage spills at
    // D = 128; zeros in the place of such blocks' V, read through a selected
    // address, took 1.3% more on 8 x 2048 tokens, where leaving them out takes
    // 0.5% less.)
    auto step = [&](auto more, auto all, int t) {
        constexpr bool kMore = decltype(more)::value;
        constexpr bool kAll = decltype(all)::value;
        if constexpr (kMore) {
            stage_v<D>(a, s_v[(t + 1) & 1], w, b_1, kvh, lane);
            if (t + 2 < nsteps) {
                b_2 = block_of(t + 2, ok_2);
                stage_k<D>(a, s_k[t & 1], w, b_2, kvh, lane);
            }
        }
        const int base = 64 * t;
        {
            // Score i of tile T: key base + 32 T + 16 (i / 8) + 8 h + i % 8.
            if (base + 63 > tq0 || ok_t != 15) [[unlikely]] {
#pragma unroll
                for (int T = 0; T < 2; ++T) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const int key = base + 32 * T + 16 * (i >> 3) + 8 * h + (i & 7);
                        if (key >= lim || !((ok_t >> (2 * T + (i >> 3))) & 1)) sc[T][i] = -INFINITY;
                    }
                }
            }
            float bm = max3(max3(sc[0][0], sc[0][1], sc[0][2]), max3(sc[0][3], sc[0][4], sc[0][5]), sc[0][6]);
#pragma unroll
            for (int i = 7; i < 31; i += 2) bm = max3(bm, sc[i >> 4][i & 15], sc[(i + 1) >> 4][(i + 1) & 15]);
            bm = max2(bm, sc[1][15]);
            {
                float x, y;
                swap32(bm, x, y);
                bm = max2(x, y) * a.scale_log2;
            }
            if (__any(bm > m + kLazyMargin)) {
                const float m_new = fmaxf(m, bm);
                const float alpha = rescale(m, m_new);
#pragma unroll
                for (int i = 0; i < ND; ++i) acc[i] *= alpha;
                l *= alpha;
                m = m_new;
            }
            const float c = ((m == -INFINITY) ? 0.0f : m) - kPExpLazy;
            f16x sn[2];
            if constexpr (kMore) qk_stage<D>(sn, s_k[(t + 1) & 1] + koff, q);
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                if (!kAll && 4 * t + b >= nvis) break;
                float p[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[b >> 1][8 * (b & 1) + i], a.scale_log2, -c));
                }
                l += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
                h2 hh[4], ll[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    hh[i] = __builtin_amdgcn_cvt_pkrtz(p[2 * i], p[2 * i + 1]);
                    ll[i] = __builtin_amdgcn_cvt_pkrtz(sub_h2_lo(p[2 * i], hh[i]), sub_h2_hi(p[2 * i + 1], hh[i]));
                }
                const h8 ph = __builtin_bit_cast(h8, __builtin_shufflevector(
                    __builtin_shufflevector(hh[0], hh[1], 0, 1, 2, 3), __builtin_shufflevector(hh[2], hh[3], 0, 1, 2, 3),
                    0, 1, 2, 3, 4, 5, 6, 7));
                const h8 pl = __builtin_bit_cast(h8, __builtin_shufflevector(
                    __builtin_shufflevector(ll[0], ll[1], 0, 1, 2, 3), __builtin_shufflevector(ll[2], ll[3], 0, 1, 2, 3),
                    0, 1, 2, 3, 4, 5, 6, 7));
                const f16* const vl = s_v[t & 1] + b * St::kTile + 8 * lane;
                h8 v[ND];
#pragma unroll
                for (int i = 0; i < ND; ++i) v[i] = *reinterpret_cast<const h8*>(vl + 512 * i);
#pragma unroll
                for (int i = 0; i < ND; ++i) acc[i] = mfma32(v[i], ph, acc[i]);
#pragma unroll
                for (int i = 0; i < ND; ++i) acc[i] = mfma32(v[i], pl, acc[i]);
            }
            if constexpr (kMore) {
                sc[0] = sn[0];
                sc[1] = sn[1];
            }
        }
        if constexpr (kMore) {
            wait_vm<0>();
            const int nv = tokens_of(t + 1, ok_1);
            if (nv < kBlockTokens) clean_v<D>(s_v[(t + 1) & 1], w, nv, lane);
            ok_t = ok_1;
            ok_1 = ok_2;
            b_1 = b_2;
            __syncthreads();
        }
    };
    int t = 0;
    for (const int whole = min(nvis / 4, nsteps - 1); t < whole; ++t) step(std::true_type{}, std::true_type{}, t);
    for (; t + 1 < nsteps; ++t) step(std::true_type{}, std::false_type{}, t);
    step(std::false_type{}, std::false_type{}, t);

    // The wave's output rows, through its quarter of the K buffers (every
    // wave's last scores are made): chunk c (8 values) of row r at chunk
    // c ^ (r % (D / 8)), so that neither side conflicts, and back as whole rows,
    // D / 8 lanes each.
    {
        float y0, y1;
        swap32(l, y0, y1);
        const float sum = y0 + y1;
        const float inv = (sum > 0.0f) ? 1.0f / sum : 0.0f;
        constexpr int kChunks = D / 8;
        f16* const o_lds = &s_k[0][0] + w * 32 * D;
#pragma unroll
        for (int i = 0; i < ND; ++i) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                h4 o;
#pragma unroll
                for (int c = 0; c < 4; ++c) o[c] = static_cast<f16>(acc[i][4 * k + c] * inv);
                *reinterpret_cast<h4*>(o_lds + r * D + 8 * ((4 * i + k) ^ (r & (kChunks - 1))) + 4 * h) = o;
            }
        }
        f16* const op = a.out + (static_cast<size_t>(start) + tq0) * a.H * D + 8 * (lane & (kChunks - 1));
        int to[D / 16];
        h8 v[D / 16];
#pragma unroll
        for (int i = 0; i < D / 16; ++i) {
            const int row = (64 / kChunks) * i + lane / kChunks;
            to[i] = __shfl(rel, row);
            v[i] = *reinterpret_cast<const h8*>(o_lds + row * D + 8 * ((lane ^ row) & (kChunks - 1)));
        }
        if (a.out16) {
#pragma unroll
            for (int i = 0; i < D / 16; ++i) {
                if (to[i] >= 0) __builtin_nontemporal_store(v[i], reinterpret_cast<h8*>(op + static_cast<size_t>(to[i]) * D));
            }
        } else {
#pragma unroll
            for (int i = 0; i < D / 16; ++i) {
                h4* const o = reinterpret_cast<h4*>(op + static_cast<size_t>(to[i]) * D);
                if (to[i] >= 0) {
                    o[0] = __builtin_shufflevector(v[i], v[i], 0, 1, 2, 3);
                    o[1] = __builtin_shufflevector(v[i], v[i], 4, 5, 6, 7);
                }
            }
        }
    }
    }
}

int prefill(const char* who, void* out, const void* q, const void* kc, const void* vc,
            const int* slots, const int* ctx, float scale, long long S, long long H, long long Hkv,
            long long D, long long BS, long long max_len, int num_blocks, hipStream_t stream) {
    if (S < 0 || H <= 0 || Hkv <= 0 || D <= 0 || BS <= 0 || max_len < 0) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER,
                    "%s: num_seqs=%lld num_heads=%lld num_kv_heads=%lld head_dim=%lld "
                    "block_size=%lld max_context_len=%lld", who, S, H, Hkv, D, BS, max_len);
    }
    if (H % Hkv != 0) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: num_heads %lld not a multiple of num_kv_heads %lld",
                    who, H, Hkv);
    }
    if ((D != 64 && D != 128) || BS != kBlockTokens) {
        return fail(SWIFTLLM_ERR_NOT_SUPPORTED, "%s: head_dim=%lld block_size=%lld (supported: 64/128, 16)",
                    who, D, BS);
    }
    if (S > 65535 || H > 65535 || max_len > (1LL << 30)) {
        return fail(SWIFTLLM_ERR_NOT_SUPPORTED, "%s: num_seqs=%lld num_heads=%lld max_context_len=%lld",
                    who, S, H, max_len);
    }
    if (S > 0 && max_len > 0 && (!out || !q || !kc || !vc || !slots || !ctx)) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: null pointer", who);
    }
    if (!aligned(out, 8) || !aligned(q, 8) || !aligned(kc, 8) || !aligned(vc, 8) ||
        !aligned(slots, 4) || !aligned(ctx, 4)) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: misaligned pointer", who);
    }
    // Workgroups per (sequence, kv head chunk): x = 8 of them per XCD round
    // times 64 * kPrefillWaves threads must stay below 2^32 threads.
    const long long G = H / Hkv;
    const long long tpw = 16 / (G < 16 ? G : 16);
    const long long per_wg = static_cast<long long>(kPrefillWaves) * 2 * tpw;
    const long long groups = (max_len + per_wg - 1) / per_wg;
    if (groups >= (1LL << 21)) {
        return fail(SWIFTLLM_ERR_NOT_SUPPORTED,
                    "%s: max_context_len=%lld needs %lld workgroups per sequence (limit 2^21)", who,
                    max_len, groups);
    }
    int rc = require_device();
    if (rc != SWIFTLLM_OK) return rc;
    if (S == 0 || max_len == 0) return ok();
    PrefillArgs a{};
    a.out = static_cast<f16*>(out);
    a.q = static_cast<const f16*>(q);
    a.kc = static_cast<const f16*>(kc);
    a.vc = static_cast<const f16*>(vc);
    a.slots = slots;
    a.ctx = ctx;
    a.scale_log2 = static_cast<float>(static_cast<double>(scale) * static_cast<double>(kLog2e));
    a.S = static_cast<int>(S);
    a.H = static_cast<int>(H);
    a.Hkv = static_cast<int>(Hkv);
    a.G = a.H / a.Hkv;
    a.nhc = (a.G + 15) / 16;
    a.gw = a.G < 16 ? a.G : 16;
    a.tpw = 16 / a.gw;
    a.groups = static_cast<int>(groups);
    a.units = S * static_cast<long long>(a.Hkv) * a.nhc;
    a.num_blocks = num_blocks;
    const long long rounds = (a.units + 7) / 8;
    const long long gy = rounds < 65535 ? rounds : 65535;
    const dim3 grid(static_cast<unsigned>(8 * a.groups), static_cast<unsigned>(gy),
                    static_cast<unsigned>((rounds + gy - 1) / gy));
    const dim3 block(64 * kPrefillWaves);
    const bool fold = a.scale_log2 > 0.0f;
    const int wide_gw = a.G < 32 ? a.G : 32;
    const int wide_heads = a.Hkv * ((a.G + 31) / 32);
    const long long wide_per = static_cast<long long>(kPrefillWaves) * (32 / wide_gw);
    const long long items = S * wide_heads * ((max_len + wide_per - 1) / wide_per);
    const long long resident = kSharedCUs * (D == 128 ? kSharedPerCU<128> : kSharedPerCU<64>);
    const bool brief = max_len * a.G <= (items <= resident ? kBriefRows : brief_rows_many(a.G, static_cast<int>(D)));
    if (fold && !brief && S <= kSharedMaxSeqs && items < (1LL << 30) && aligned(kc, 16) && aligned(vc, 16)) {
        a.nhc = (a.G + 31) / 32;
        a.gw = wide_gw;
        a.tpw = 32 / wide_gw;
        a.groups = static_cast<int>((max_len + wide_per - 1) / wide_per);
        const int heads = wide_heads;
        a.xcds = heads % 8 == 0 ? 8 : 1;
        a.q16 = aligned(q, 16);
        a.out16 = aligned(out, 16);
        const long long wgs = std::min<long long>((items + 7) / 8 * 8, resident);
        return launched(launch(D == 128 ? paged_prefill_shared_kernel<128> : paged_prefill_shared_kernel<64>,
                               dim3(static_cast<unsigned>(wgs)), block, 0, stream, a),
                        who);
    }
    const bool ldsk = aligned(kc, 16);
    using K = void (*)(PrefillArgs);
    static const K kernels[2][2][2] = {
        {{paged_prefill_kernel<64, false, false>, paged_prefill_kernel<64, false, true>},
         {paged_prefill_kernel<64, true, false>, paged_prefill_kernel<64, true, true>}},
        {{paged_prefill_kernel<128, false, false>, paged_prefill_kernel<128, false, true>},
         {paged_prefill_kernel<128, true, false>, paged_prefill_kernel<128, true, true>}}};
    const hipError_t err =
        launch(kernels[D == 128][fold][ldsk], grid, block, 0, stream, a);
    return launched(err, who);
}

}  // namespace
}  // namespace swiftllm

using namespace swiftllm;

extern "C" {

int swiftllm_hip_paged_attention_prefill(void* output, const void* query, const void* key_cache,
                                         const void* value_cache, const int32_t* slot_mapping,
                                         const int32_t* context_lens,
                                         const swiftllm_paged_attention_params* p,
                                         hipStream_t stream) {
    const char* who = "swiftllm_hip_paged_attention_prefill";
    if (p == nullptr) return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: null params", who);
    const size_t lim = 0x7fffffff;
    if (p->num_seqs > lim || p->num_heads > lim || p->num_kv_heads > lim || p->head_dim > lim ||
        p->block_size > lim || p->max_context_len > lim) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: parameter out of range", who);
    }
    return prefill(who, output, query, key_cache, value_cache, slot_mapping, context_lens, p->scale,
                   static_cast<long long>(p->num_seqs), static_cast<long long>(p->num_heads),
                   static_cast<long long>(p->num_kv_heads), static_cast<long long>(p->head_dim),
                   static_cast<long long>(p->block_size), static_cast<long long>(p->max_context_len),
                   0, stream);
}

int swiftllm_hip_launch_paged_prefill(void* output, const void* query, const void* key_cache,
                                      const void* value_cache, const int32_t* slot_mapping,
                                      const int32_t* context_lens, float scale, int num_seqs,
                                      int num_heads, int num_kv_heads, int head_dim, int block_size,
                                      int max_context_len, int num_blocks, hipStream_t stream) {
    return prefill("swiftllm_hip_launch_paged_prefill", output, query, key_cache, value_cache,
                   slot_mapping, context_lens, scale, num_seqs, num_heads, num_kv_heads, head_dim,
                   block_size, max_context_len, num_blocks, stream);
}

}  // extern "C"
