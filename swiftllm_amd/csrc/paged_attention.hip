// Paged-attention decode for gfx950 (CDNA4).
//
// Contract (paged_attention.cu:35-137 is the reference's text; its output
// stage is a stub, so the behaviour below is the textbook attention its
// comments and indexing describe):
//   for sequence s, query head h, kv head kvh = h / (H / Hkv)   (cu:52)
//   L = context_lens[s]; token j lives in block bt[s, j / 16] at offset j % 16
//   logit_j = scale * sum_d q[s,h,d] * K(b, kvh, d, j % 16)     (cu:92-96)
//   out[s,h,:] = sum_j softmax(logit)_j * V(b, kvh, :, j % 16)  (cu:113-135)
// fp16 in and out, fp32 accumulation; L <= 0 writes zeros.
//
// Work decomposition. One workgroup serves every query head of one kv head
// (up to 16 per workgroup), so each K/V tile is read from HBM once. The
// reference grid (S, H) (cu:248) re-reads it H/Hkv times. The waves of a
// workgroup take the blocks of its token range round-robin; the range is the
// whole context (single pass) or one partition of it (split-K). Each wave
// keeps a running max, sum and output for its blocks; the waves merge through
// LDS. Split-K partitions leave (max, sum, output) in a workspace and a
// second kernel does the rescaled reduce (the kernel boundary makes the
// partials visible; an in-kernel last-arriver reduce would need device-scope
// fences, which write back and invalidate the whole L2 on this GPU).
//
// Per 16-token block, each wave runs the whole computation on the matrix
// cores with v_mfma_f32_16x16x16_f16 (the group of query heads is the N = 16
// side, zero-padded):
//   1. K tile rows 16J..16J+15 arrive with tokens contiguous ([d][t]); an
//      MFMA against a 0/1 identity operand returns the same values in the
//      transposed ([t][d]) register layout, exactly (one product per output).
//   2. S^T[t][g] = sum_d K^T[t][d] Q^T[d][g]          (D/16 MFMAs)
//   3. Online softmax in fp32 on the S^T accumulator; the 4 token rows of a
//      head live in lanes l, l^16, l^32, l^48, so the block max is two xor
//      shuffles.
//   4. O^T[d][g] += V[d][t] P^T[t][g] with V in its stored layout. P is fed as
//      an fp16 hi part plus an fp16 lo part (two MFMAs), which keeps ~22 bits
//      of each probability; P is computed as 2^15 * exp2(s - m) so both parts
//      stay in fp16's normal range.

#include <algorithm>
#include <cmath>
#include <mutex>

#include "attention_core.hpp"

namespace swiftllm {
namespace {

using namespace attn;

struct DecodeArgs {
    f16* out;
    const f16* q;
    const f16* kc;
    const f16* vc;
    const int* bt;
    const int* ctx;
    float* ws_max;       // [S][H][MP]         log2-domain max logit
    float* ws_sum;       // [S][H][MP]         sum of 2^15 * exp2(s - max)
    float* ws_out;       // [S][H][MP][D]      normalised partial output
    float scale_log2;    // scale * log2(e)
    int H;
    int Hkv;
    int G;            // query heads per kv head
    int nhc;          // head chunks of 16 per kv head
    int MB;           // max_num_blocks_per_seq (row stride of bt)
    int num_blocks;   // bound on block ids; <= 0: unbounded
    int part_blocks;  // blocks per partition; 0: single pass
    int MP;           // partitions per sequence in the workspace
    int S;            // sequences
    float share;      // split-K items: kItemShare of a resident workgroup, per block of the batch
    bool single;      // the partition kernel runs a single-pass call
    int snake;        // > 0: single-pass item order in snake rounds of this many
};

// Attends `count` blocks of one sequence: logical blocks first,
// first + stride, ... Blocks are double-buffered in registers, so the next
// block's loads are in flight while one is attended. The steady-state loop
// runs while at least three blocks are left: both of its loads are real
// blocks, no load depends on a condition, and the compiler's wait counts stay
// exact. The last one or two blocks are peeled off, so no tile is read twice.
template <int D>
__device__ __forceinline__ void attend_blocks(WaveState<D>& st, const const_int* btrow, int first,
                                              int stride, int count, int L, const f16* kc,
                                              const f16* vc, int Hkv, int num_blocks, int kvh,
                                              int loff, int kg, const QOperand<D>& qB, h4 ident,
                                              float scale_log2) {
    constexpr int NJ = D / 16;
    if (count <= 0) return;
    auto block_at = [&](int j) { return __builtin_amdgcn_readfirstlane(btrow[j]); };
    auto valid_of = [&](int j, int b) {
        return block_ok(b, num_blocks) ? min(kBlockTokens, L - j * kBlockTokens) : 0;
    };
    h4 kA[NJ], vA[NJ], kB[NJ], vB[NJ];
    int jA = first;
    int bA = block_at(jA);
    load_tile<D>(kc, vc, Hkv, num_blocks, bA, kvh, loff, kA, vA);
    int left = count;
    for (; left > 2; left -= 2) {
        const int jB = jA + stride;
        const int bB = block_at(jB);
        load_tile<D>(kc, vc, Hkv, num_blocks, bB, kvh, loff, kB, vB);
        attend_block<D>(st, valid_of(jA, bA), kg, kA, vA, qB, ident, scale_log2);
        jA = jB + stride;
        bA = block_at(jA);
        load_tile<D>(kc, vc, Hkv, num_blocks, bA, kvh, loff, kA, vA);
        attend_block<D>(st, valid_of(jB, bB), kg, kB, vB, qB, ident, scale_log2);
    }
    if (left == 2) {
        const int jB = jA + stride;
        const int bB = block_at(jB);
        load_tile<D>(kc, vc, Hkv, num_blocks, bB, kvh, loff, kB, vB);
        attend_block<D>(st, valid_of(jA, bA), kg, kA, vA, qB, ident, scale_log2);
        attend_block<D>(st, valid_of(jB, bB), kg, kB, vB, qB, ident, scale_log2);
    } else {
        attend_block<D>(st, valid_of(jA, bA), kg, kA, vA, qB, ident, scale_log2);
    }
}

// The sequence with the r-th longest context (ties by index) of at most
// kLptMaxSeqs, found by every workgroup of a single-pass grid that is resident all at once (the snake
// order below). Each thread ranks S / 256 sequences against all S, so the
// cost grows as S^2: measured on MI355X with the ranking in every grid,
// 1024 sequences of 32-128 tokens took 1324 us against 67 us in plain order,
// and 256 of them 39.7 against 18.8 us. So only batches of up to
// kLptMaxSeqs sequences are ranked (at most 128 compares a thread), and larger
// grids run in sequence order, which the dispatcher balances as workgroups
// finish.
constexpr int kLptMaxSeqs = 128;

__device__ __forceinline__ int sequence_for_block(const int* ctx, int S, int r) {
    __shared__ int s_ctx[kLptMaxSeqs];
    __shared__ int s_seq;
    for (int c = threadIdx.x; c < S; c += blockDim.x) s_ctx[c] = ctx[c];
    if (threadIdx.x == 0) s_seq = r;
    __syncthreads();
    for (int c = threadIdx.x; c < S; c += blockDim.x) {
        const int lc = s_ctx[c];
        int rank = 0;
        for (int o = 0; o < S; ++o) {
            const int lo = s_ctx[o];
            rank += (lo > lc) || (lo == lc && o < c);
        }
        if (rank == r) s_seq = c;
    }
    __syncthreads();
    return s_seq;
}

// Dynamic LDS of decode_item's wave merge, in floats: per wave 16 maxima,
// 16 sums and gstride = min(G, 16) rows of D partial outputs.
template <int D, int NW>
__host__ __device__ constexpr int merge_lds_floats(int G) {
    return NW * 32 + NW * (G < 16 ? G : 16) * D;
}

// Merges the NW waves' running states of one item through LDS and hands every
// normalised output to emit(g, d, o, M, den): query head g of the gn served
// here, dimension d, with the merged max and sum. l_run: the wave's sum over
// its four lane groups.
template <int D, int NW, typename Emit>
__device__ __forceinline__ void merge_waves(float* smem, const WaveState<D>& st, float l_run, int gn,
                                            int gstride, int w, int r, int kg, Emit emit) {
    float* sm_m = smem;            // [NW][16]
    float* sm_l = smem + NW * 16;  // [NW][16]
    float* sm_o = smem + NW * 32;  // [NW][gstride][D]
    if (kg == 0) {
        sm_m[w * 16 + r] = st.m;
        sm_l[w * 16 + r] = l_run;
    }
    if (r < gn) {
#pragma unroll
        for (int J = 0; J < D / 16; ++J) {
            *reinterpret_cast<f4*>(sm_o + static_cast<size_t>(w * gstride + r) * D + 16 * J + 4 * kg) = st.acc[J];
        }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < gn * D; idx += NW * 64) {
        const int g = idx / D;
        const int d = idx - g * D;
        float M = -INFINITY;
#pragma unroll
        for (int w2 = 0; w2 < NW; ++w2) M = fmaxf(M, sm_m[w2 * 16 + g]);
        float num = 0.0f, den = 0.0f;
#pragma unroll
        for (int w2 = 0; w2 < NW; ++w2) {
            const float mw = sm_m[w2 * 16 + g];
            const float f = (mw == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(mw - M);
            num += f * sm_o[static_cast<size_t>(w2 * gstride + g) * D + d];
            den += f * sm_l[w2 * 16 + g];
        }
        emit(g, d, (den > 0.0f) ? num / den : 0.0f, M, den);
    }
}

// Bytes of the partition kernel's item list for S sequences (int prefix of
// S + 1 entries, 17 int counts per group of 64 sequences, 16-bit sequence list
// of S), rounded to 16.
__host__ __device__ constexpr size_t part_list_lds_bytes(int S) {
    return ((static_cast<size_t>(S) + 1) * 4 + (static_cast<size_t>(S) + 63) / 64 * 17 * 4 +
            static_cast<size_t>(S) * 2 + 15) / 16 * 16;
}

// One (sequence, kv head, head chunk, partition) item. The NW waves of the
// workgroup take the item's blocks round-robin and merge through LDS; the
// result is the output (single pass, or a sequence with one partition) or a
// split-K partial. Every thread of the workgroup calls it with the same item.
// `len`: the sequence's context length where the caller has it, else -1.
template <int D, int NW>
__device__ __forceinline__ void decode_item(const DecodeArgs& a, int s, int kvh, int hc,
                                            int part, int part_blocks, int len = -1) {
    constexpr int NJ = D / 16;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15;   // MFMA column / row-in-slice index
    const int kg = lane >> 4;  // MFMA k-group: 4 consecutive k per lane

    const int g0 = hc * 16;
    const int gn = min(16, a.G - g0);  // query heads served here
    const int gstride = min(16, a.G);  // LDS rows per wave
    const int h0 = kvh * a.G + g0;

    int L = len;
    if (len < 0) L = max(a.ctx[s], 0);
    const int nblk = min((L + kBlockTokens - 1) / kBlockTokens, a.MB);
    L = min(L, nblk * kBlockTokens);
    int nparts, jb0, jb1;
    if (part_blocks > 0) {
        nparts = (nblk + part_blocks - 1) / part_blocks;
        jb0 = part * part_blocks;
        jb1 = min(nblk, jb0 + part_blocks);
    } else {
        nparts = 1;
        jb0 = 0;
        jb1 = nblk;
    }
    if (nblk == 0) {
        if (part == 0) {
            for (int i = threadIdx.x; i < gn * D; i += NW * 64) {
                a.out[(static_cast<size_t>(s) * a.H + h0) * D + i] = static_cast<f16>(0.0f);
            }
        }
        return;
    }
    if (part >= nparts) return;

    QOperand<D> qB;
    {
        const f16* qp = a.q + (static_cast<size_t>(s) * a.H + h0 + min(r, gn - 1)) * D + 4 * kg;
#pragma unroll
        for (int J = 0; J < NJ; ++J) {
            const h4 v = *reinterpret_cast<const h4*>(qp + 16 * J);
            qB.v[J] = (r < gn) ? v : h4{0, 0, 0, 0};
        }
    }
    // Identity operand of step 1: B[k = 4kg + i][n = r] = (k == n).
    h4 ident;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        ident[i] = (4 * kg + i == r) ? static_cast<f16>(1.0f) : static_cast<f16>(0.0f);
    }
    // Lane (r, kg) loads tile row 16J + r, tokens 4kg .. 4kg + 3.
    const int loff = kv_elem_offset(r, 4 * kg);
    const const_int* btrow = as_const(a.bt) + static_cast<size_t>(s) * a.MB;

    WaveState<D> st;
    st.m = -INFINITY;
    st.l = 0.0f;
#pragma unroll
    for (int J = 0; J < NJ; ++J) st.acc[J] = f4{0, 0, 0, 0};

    // Blocks jb0 + w, jb0 + w + NW, ... of this wave.
    const int first = jb0 + w;
    const int nbw = (jb1 > first) ? (jb1 - first + NW - 1) / NW : 0;
    attend_blocks<D>(st, btrow, first, NW, nbw, L, a.kc, a.vc, a.Hkv, a.num_blocks, kvh, loff, kg,
                     qB, ident, a.scale_log2);
    // Per-lane partial sums cover tokens 4kg..4kg+3 of every block.
    const float l_run = sum_over_kg(st.l);
    extern __shared__ __align__(16) float smem[];
    merge_waves<D, NW>(smem, st, l_run, gn, gstride, w, r, kg, [&](int g, int d, float o, float M, float den) {
        const int h = h0 + g;
        if (nparts == 1) {
            a.out[(static_cast<size_t>(s) * a.H + h) * D + d] = static_cast<f16>(o);
        } else {
            const size_t pi = (static_cast<size_t>(s) * a.H + h) * a.MP + part;
            a.ws_out[pi * D + d] = o;
            if (d == 0) {
                a.ws_max[pi] = M;
                a.ws_sum[pi] = den;
            }
        }
    });
}

// At least two waves per SIMD: caps the registers (at 157 VGPRs for D=128 the
// kernel fits three waves per SIMD), so several workgroups share a CU.
template <int D, int NW>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(2)))
void paged_decode_kernel(const DecodeArgs a) {
    int kvh, hc, s;
    if (a.snake > 0) {
        // Single pass, whole grid resident: workgroup i takes item
        // snake(i) of the longest-first list of (sequence, kv head, head
        // chunk) items, where the list is cut into rounds of `snake`
        // items and every other round runs backwards. Workgroups i and
        // i + snake, which the dispatcher puts on the same CU, then pair a
        // long sequence with a short one.
        const int HC = gridDim.y;
        const int i = blockIdx.z * HC + blockIdx.y;
        const int k = i / a.snake;
        const int pos = i - k * a.snake;
        const int rlen = min(a.snake, static_cast<int>(gridDim.z) * HC - k * a.snake);
        const int item = k * a.snake + ((k & 1) ? (rlen - 1 - pos) : pos);
        const int sub = item % HC;
        kvh = sub / a.nhc;
        hc = sub - kvh * a.nhc;
        s = sequence_for_block(a.ctx, gridDim.z, item / HC);
    } else {
        kvh = blockIdx.y / a.nhc;
        hc = blockIdx.y - kvh * a.nhc;
        s = blockIdx.z;
    }
    decode_item<D, NW>(a, s, kvh, hc, 0, 0);
}

// Split-K partitions. The items are the real (sequence, partition) pairs
// times the kv-head chunks, longest first: every workgroup lists them in LDS
// and walks items blockIdx.x, + gridDim.x, ... The grid is sized to the
// resident workgroups, not to the worst case of every sequence, so a ragged
// batch launches no empty workgroups (a grid over max_num_blocks_per_seq
// would be mostly empty). Workgroups start in blockIdx order, so the order of
// the list is the order the items start in: first every full partition (of
// item_blocks() blocks), then the last, partial partition of each sequence in
// kLptClasses length classes, longest first (an empty sequence's item, which
// writes zeros, is a partial of length 0). A single-pass call of several rounds
// may take the same list with one partition per sequence (list_pays). Measured
// with the gather kernel of libswiftllm_ceilings on config 4's items at
// 1024-token partitions: 151 us longest first against 166 us in sequence order.
//
// The item of one list position is run by several workgroups (one per kv-head
// chunk), each with its own copy of the list, so the list must come out the
// same in every workgroup: within a class the partials keep sequence order,
// placed by prefix sums, never by the order atomics happen to land in. The
// list costs every workgroup a prologue, so it is built with one wave per
// group of 64 sequences, class counts and ranks by ballots and sums by DPP,
// three barriers in all; with a shuffle scan of packed class counts per chunk
// of 256 sequences, 256 contexts of 16-128 tokens took 31.8 us instead of 27.9,
// lognormal ones up to 8192 tokens 181.9 instead of 175.9.
// Batches of more than kPartMaxSeqs sequences take one item per workgroup
// over the full grid.
constexpr int kPartMaxSeqs = 4096;
constexpr int kLptClasses = 16;

// Blocks per item of this batch: as many whole partitions as fit in kItemShare
// times a resident workgroup's share of all blocks, at least one. Short items
// pay a start-up and a merge each, long ones leave a tail; longest first, an
// item of about one share starts early enough. Measured at 512-token
// partitions (us per call, 256 lognormal contexts up to 8192 tokens, 32/8
// heads x 128): one partition per item 197, items of half a share 190, of one
// 183.6, of one and a half 181.9, of two 181.7 (150 contexts of 64/8 heads:
// 146, 133, 130, 129; 256 of 1000-4000 tokens: 406, 396, 398, 402). Every
// workgroup of the partition kernel and every wave of its reduce works it out
// for itself, from the lengths alone.
constexpr float kItemShare = 1.5f;

// Blocks of the batch's contexts, each counted as 2^18 (4M tokens) at most, so
// that kPartMaxSeqs of them fit in an int; every wave works them out for itself.
struct BatchBlocks {
    int sum, longest;
    int len;  // context length of sequence `s`
};

__device__ __forceinline__ BatchBlocks batch_blocks(const int* ctx, int S, int MB, int s) {
    BatchBlocks b{0, 0, 0};
    const int cap = min(MB, 1 << 18);
#pragma unroll 4
    for (int i = threadIdx.x & 63; i < S; i += 64) {
        const int len = max(ctx[i], 0);
        const int n = min((len + kBlockTokens - 1) / kBlockTokens, cap);
        b.sum += n;
        b.longest = max(b.longest, n);
        b.len = (i ^ s) < 64 ? len : b.len;  // lanes of s's group of 64
    }
    return BatchBlocks{wave_total(b.sum), wave_max(b.longest), __builtin_amdgcn_readlane(b.len, s & 63)};
}

__device__ __forceinline__ int item_blocks(const int* ctx, int S, int MB, int part_blocks, float share) {
    const int sum = batch_blocks(ctx, S, MB, 0).sum;
    const int most = static_cast<int>(fminf(static_cast<float>(sum) * share, 0x1p28f));
    return __builtin_amdgcn_readfirstlane(part_blocks * max(1, most / part_blocks));
}

// Whether a single-pass batch is run through the list (one item per sequence,
// longest first) or in plain order. The table's width says nothing of the
// contexts, so the kernel looks at them. Plain order ends later than the list
// by the time its longest context still takes once the others are done, at
// most its chain and at most the batch's time; the list costs every workgroup
// its prologue, about 0.04 us per sequence. So: a longest context of some
// length for the number of sequences, work enough before it, and well above the
// mean. Measured (us per call, plain / list, tables 512 blocks wide): 256
// lognormal contexts, 32/8 heads x 128, 227 / 198; 96, 16/16 x 128, 118 / 102;
// 128 of 64-1024 tokens, 32/8 x 128, 54.5 / 52.6, 8/8 x 64 25.9 / 28.4; 256 of
// 16-128 17.0 / 27.4, 8/8 x 64 9.3 / 17.5; 1024 of 16-128 63.6 / 102.5; 127 of
// 32 beside one of 2500, 8/8 x 64, 19.9 / 21.9; 128 of 1024 80.0 / 82.1.
template <int D>
__device__ __forceinline__ bool list_pays(BatchBlocks b, int S, int HC) {
    return b.longest * (D / 64) > 2 * (S / 4 + 16) && static_cast<float>(b.sum) * HC > 32.0f * S &&
           2.0f * b.longest * S > 3.0f * b.sum;
}

template <int D, int NW>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(3)))
void paged_partition_kernel(const DecodeArgs a) {
    const int HC = a.Hkv * a.nhc;
    if (a.S > kPartMaxSeqs) {
        const int it = blockIdx.x;
        const int part = it % a.MP;
        const int sub = (it / a.MP) % HC;
        const int s = it / (a.MP * HC);
        if (s < a.S) decode_item<D, NW>(a, s, sub / a.nhc, sub % a.nhc, part, a.part_blocks);
        return;
    }
    // The item list sits in dynamic LDS after decode_item's merge area, sized
    // by the host for this batch (part_list_lds_bytes): s_pre[S + 1] exclusive
    // prefix of full partitions, s_cnt[groups of 64][kLptClasses + 1] partials
    // per class and full partitions of each group, s_part[S] sequences with a
    // partial partition, longest first.
    extern __shared__ __align__(16) float smem[];
    constexpr int kCols = kLptClasses + 1;
    const int ngroups = (a.S + 63) / 64;
    int* s_pre = reinterpret_cast<int*>(smem + merge_lds_floats<D, NW>(a.G));
    int* s_cnt = s_pre + a.S + 1;
    unsigned short* s_part = reinterpret_cast<unsigned short*>(s_cnt + ngroups * kCols);
    __shared__ int s_total[2];  // full partitions, partial ones
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (a.single) {
        int sq = blockIdx.x / HC;
        BatchBlocks b = batch_blocks(a.ctx, a.S, a.MB, sq);
        if (!list_pays<D>(b, a.S, HC)) {
            for (int it = blockIdx.x; it < a.S * HC; it += gridDim.x) {
                sq = it / HC;
                const int sub = it - sq * HC;
                decode_item<D, NW>(a, sq, sub / a.nhc, sub % a.nhc, 0, 0, b.len);
                b.len = -1;
                __syncthreads();  // the item's LDS is free again
            }
            return;
        }
    }
    const int pb = item_blocks(a.ctx, a.S, a.MB, a.part_blocks, a.share);
    // Blocks of sequence 64 * group + lane, -1 past the batch.
    auto nblk_of = [&](int group) {
        const int sq = 64 * group + lane;
        return sq < a.S ? min((max(a.ctx[sq], 0) + kBlockTokens - 1) / kBlockTokens, a.MB) : -1;
    };
    // Class of a sequence's partial partition (0 = longest), or -1 when its
    // last partition is full.
    auto class_of = [&](int nblk) {
        const int rem = nblk - (nblk / pb) * pb;
        if (nblk < 0 || (rem == 0 && nblk > 0)) return -1;
        // rem < pb <= 2^28
        return kLptClasses - 1 - static_cast<int>(static_cast<unsigned>(rem) * kLptClasses / static_cast<unsigned>(pb));
    };
    // Counts per group of 64 sequences, one wave per group: lane k gets class
    // k's from a ballot.
    for (int gr = w; gr < ngroups; gr += NW) {
        const int nblk = nblk_of(gr);
        const int c = class_of(nblk);
        const int full = wave_total(max(nblk, 0) / pb);
        int n = full;
#pragma unroll
        for (int k = 0; k < kLptClasses; ++k) {
            const int nk = __popcll(__ballot(c == k));
            if (lane == k) n = nk;
        }
        if (lane < kCols) s_cnt[gr * kCols + lane] = n;
    }
    __syncthreads();
    // Exclusive prefixes down the groups, then the classes' first positions
    // on top (lane k: class k; lane kLptClasses: full partitions).
    if (w == 0) {
        int run = 0;
        if (lane < kCols) {
            for (int gr = 0; gr < ngroups; ++gr) {
                const int n = s_cnt[gr * kCols + lane];
                s_cnt[gr * kCols + lane] = run;
                run += n;
            }
        }
        const int mine = lane < kLptClasses ? run : 0;
        const int incl = wave_inclusive_scan(mine);
        if (lane < kLptClasses) {
            for (int gr = 0; gr < ngroups; ++gr) s_cnt[gr * kCols + lane] += incl - mine;
        }
        if (lane == kLptClasses) s_total[0] = run;
        if (lane == 63) s_total[1] = incl;
    }
    __syncthreads();
    // Places each sequence: its full partitions' prefix, and its partial
    // partition at its class's next position, in sequence order.
    for (int gr = w; gr < ngroups; gr += NW) {
        const int nblk = nblk_of(gr);
        const int c = class_of(nblk);
        const int v = max(nblk, 0) / pb;
        const int x = wave_inclusive_scan(v);
        if (nblk >= 0) s_pre[64 * gr + lane] = s_cnt[gr * kCols + kLptClasses] + x - v;
        unsigned long long same = 0;
#pragma unroll
        for (int k = 0; k < kLptClasses; ++k) {
            const unsigned long long m = __ballot(c == k);
            if (c == k) same = m;
        }
        if (c >= 0) {
            const int rank = __popcll(same & ((1ull << lane) - 1ull));
            s_part[s_cnt[gr * kCols + c] + rank] = static_cast<unsigned short>(64 * gr + lane);
        }
    }
    if (threadIdx.x == 0) s_pre[a.S] = s_total[0];
    __syncthreads();
    const int nfull = __builtin_amdgcn_readfirstlane(s_total[0]);
    const int total = (nfull + __builtin_amdgcn_readfirstlane(s_total[1])) * HC;
    for (int it = blockIdx.x; it < total; it += gridDim.x) {
        const int pidx = it / HC;
        const int sub = it - pidx * HC;
        int sq, part;
        if (pidx < nfull) {
            int lo = 0, hi = a.S;  // s_pre[lo] <= pidx < s_pre[hi]
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (s_pre[mid] <= pidx) lo = mid; else hi = mid;
            }
            sq = lo;
            part = pidx - s_pre[lo];
        } else {
            sq = s_part[pidx - nfull];
            part = s_pre[sq + 1] - s_pre[sq];  // after the full ones
        }
        decode_item<D, NW>(a, sq, sub / a.nhc, sub % a.nhc, part, pb);
        __syncthreads();  // the item's LDS is free again
    }
}

// Rescaled combine of P fragments of one query head: fragment p holds a max
// m_p (log2 domain), a sum l_p and a normalised partial output o_p[D], and
// out[d] = sum_p w_p o_p[d] / sum_p w_p with w_p = exp2(m_p - M) l_p,
// M = max_p m_p. Accessors: fm(p), fl(p) and fo(p) (pointer to o_p, 8-byte
// aligned); out(d, v) stores one output.
// One wave combines a head: no barriers, lane l owns outputs
// [l * D / 64, (l + 1) * D / 64), so every fragment row is one coalesced load.
// The rows of the first kReduceRows fragments are loaded before the headers
// (max and sum) of the first 64, all in flight together, so the combine pays
// one memory latency per kReduceRows fragments; rows past the last fragment
// re-read it and get weight 0. The weights live one per lane and are broadcast
// with readlane; the rows are added in fragment order.
constexpr int kReduceRows = 16;

template <int D>
__device__ __forceinline__ void load_row(const float* p, float (&v)[D / 64]) {
    if constexpr (D == 128) {
        const float2 x = *reinterpret_cast<const float2*>(p);
        v[0] = x.x;
        v[1] = x.y;
    } else {
        v[0] = *p;
    }
}

__device__ __forceinline__ float readlane_f(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

template <int D, typename FM, typename FL, typename FO, typename OUT>
__device__ __forceinline__ void combine_head_wave(int P, FM fm, FL fl, FO fo, OUT out) {
    constexpr int CH = kReduceRows;
    constexpr int DL = D / 64;
    const int lane = threadIdx.x & 63;
    if (P <= 0) {
#pragma unroll
        for (int j = 0; j < DL; ++j) out(lane * DL + j, 0.0f);
        return;
    }
    float v[CH][DL];
#pragma unroll
    for (int i = 0; i < CH; ++i) load_row<D>(fo(min(i, P - 1)) + lane * DL, v[i]);
    const float m0 = lane < P ? fm(lane) : -INFINITY;
    const float l0 = lane < P ? fl(lane) : 0.0f;
    float M = m0;
    for (int p = 64 + lane; p < P; p += 64) M = fmaxf(M, fm(p));
    M = wave_max(M);
    float acc[DL];
#pragma unroll
    for (int j = 0; j < DL; ++j) acc[j] = 0.0f;
    float den = 0.0f;
    float w = 0.0f;
    for (int c0 = 0; c0 < P; c0 += CH) {
        if ((c0 & 63) == 0) {
            // Weights of fragments c0 .. c0 + 63, fragment c0 + l on lane l.
            if (c0 == 0) {
                w = (m0 == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(m0 - M) * l0;
            } else {
                const int p = c0 + lane;
                const float mp = p < P ? fm(p) : -INFINITY;
                w = (mp == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(mp - M) * fl(p);
            }
            den += w;
        }
        if (c0 > 0) {
#pragma unroll
            for (int i = 0; i < CH; ++i) load_row<D>(fo(min(c0 + i, P - 1)) + lane * DL, v[i]);
        }
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const float wi = readlane_f(w, (c0 & 63) + i);
#pragma unroll
            for (int j = 0; j < DL; ++j) acc[j] += wi * v[i][j];
        }
    }
    den = wave_sum(den);
    const float inv = den > 0.0f ? 1.0f / den : 0.0f;
#pragma unroll
    for (int j = 0; j < DL; ++j) out(lane * DL + j, acc[j] * inv);
}

// The same combine by the NW waves of a workgroup, for heads with many
// fragments: wave w takes the 16-fragment chunks w, w + NW, ..., keeping a
// running max, sum and rescaled partial over its chunks (one memory latency
// per chunk, its 16 rows loaded before the headers), and wave 0 merges the
// NW partials through LDS. A head then costs ceil(P / (16 NW)) latencies
// instead of ceil(P / 16), with NW times the waves in flight.
template <int D, int NW, typename FM, typename FL, typename FO, typename OUT>
__device__ __forceinline__ void combine_head_split(int P, FM fm, FL fl, FO fo, OUT out) {
    constexpr int DL = D / 64;
    constexpr int CH = kReduceRows;
    __shared__ float s_acc[NW][D];
    __shared__ float s_md[NW][2];
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    if (P <= 0) {
        if (wv == 0) {
#pragma unroll
            for (int j = 0; j < DL; ++j) out(lane * DL + j, 0.0f);
        }
        return;
    }
    float M = -INFINITY;
    float den = 0.0f;
    float acc[DL];
#pragma unroll
    for (int j = 0; j < DL; ++j) acc[j] = 0.0f;
    for (int c0 = wv * CH; c0 < P; c0 += NW * CH) {
        float v[CH][DL];
#pragma unroll
        for (int i = 0; i < CH; ++i) load_row<D>(fo(min(c0 + i, P - 1)) + lane * DL, v[i]);
        const int p = c0 + lane;
        const bool mine = lane < CH && p < P;
        const float mp = mine ? fm(p) : -INFINITY;
        const float lp = mine ? fl(p) : 0.0f;
        const float Mn = fmaxf(M, wave_max(mp));
        if (Mn == -INFINITY) continue;  // every fragment so far empty (wave-uniform)
        const float sc = (M == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(M - Mn);
        const float w = (mp == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(mp - Mn) * lp;
        den = den * sc + wave_sum(w);
#pragma unroll
        for (int j = 0; j < DL; ++j) acc[j] *= sc;
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const float wi = readlane_f(w, i);
#pragma unroll
            for (int j = 0; j < DL; ++j) acc[j] += wi * v[i][j];
        }
        M = Mn;
    }
#pragma unroll
    for (int j = 0; j < DL; ++j) s_acc[wv][lane * DL + j] = acc[j];
    if (lane == 0) {
        s_md[wv][0] = M;
        s_md[wv][1] = den;
    }
    __syncthreads();
    if (wv != 0) return;
    float Mall = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) Mall = fmaxf(Mall, s_md[w][0]);
    float tot[DL];
#pragma unroll
    for (int j = 0; j < DL; ++j) tot[j] = 0.0f;
    float dall = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const float Mw = s_md[w][0];
        const float f = (Mw == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(Mw - Mall);
        dall += f * s_md[w][1];
#pragma unroll
        for (int j = 0; j < DL; ++j) tot[j] += f * s_acc[w][lane * DL + j];
    }
    const float inv = dall > 0.0f ? 1.0f / dall : 0.0f;
#pragma unroll
    for (int j = 0; j < DL; ++j) out(lane * DL + j, tot[j] * inv);
}

// Split-K reduce of the partition kernel: one wave per (query head,
// sequence); sequences with a single partition were written directly by the
// partition kernel.
struct ReduceArgs {
    f16* out;
    const int* ctx;
    const float* ws_max;
    const float* ws_sum;
    const float* ws_out;
    int S;
    int H;
    int MB;
    int part_blocks;
    int MP;
    float share;
};

// Combine of head h of sequence s by one wave, or by the four waves of the
// workgroup (SPLIT).
template <int D, bool SPLIT>
__device__ __forceinline__ void reduce_head(const ReduceArgs& a, int s, int h) {
    const int L = max(a.ctx[s], 0);
    const int nblk = min((L + kBlockTokens - 1) / kBlockTokens, a.MB);
    if (nblk <= a.part_blocks) return;
    const int pb = a.S <= kPartMaxSeqs ? item_blocks(a.ctx, a.S, a.MB, a.part_blocks, a.share) : a.part_blocks;
    const int nparts = (nblk + pb - 1) / pb;
    if (nparts <= 1) return;
    const size_t row = static_cast<size_t>(s) * a.H + h;
    const float* pm = a.ws_max + row * a.MP;
    const float* pl = a.ws_sum + row * a.MP;
    const float* po = a.ws_out + row * a.MP * D;
    f16* o = a.out + row * D;
    auto fm = [&](int p) { return pm[p]; };
    auto fl = [&](int p) { return pl[p]; };
    auto fo = [&](int p) { return po + static_cast<size_t>(p) * D; };
    auto out = [&](int d, float v) { o[d] = static_cast<f16>(v); };
    if constexpr (SPLIT) {
        combine_head_split<D, 4>(nparts, fm, fl, fo, out);
    } else {
        combine_head_wave<D>(nparts, fm, fl, fo, out);
    }
}

// One wave per (query head, sequence), four heads per workgroup.
template <int D>
__global__ __launch_bounds__(256) void paged_reduce_wave_kernel(const ReduceArgs a) {
    const int h = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (h >= a.H) return;
    reduce_head<D, false>(a, blockIdx.y, h);
}

// One (query head, sequence) per workgroup of four waves, for more than 16
// partitions per sequence.
template <int D>
__global__ __launch_bounds__(256) void paged_reduce_split_kernel(const ReduceArgs a) {
    reduce_head<D, true>(a, blockIdx.y, blockIdx.x);
}

// ---------------------------------------------------------------------------
// Balanced ("stream-K") decode. The blocks of all sequences form one list,
// sequence by sequence. A team of TS = Hkv * nhc consecutive waves (one per
// kv head and head chunk) takes blocks [t*q, (t+1)*q) of that list, with
// q = ceil(blocks / teams): every team gets the same number of blocks
// whatever the context lengths, the grid runs in one round, and the waves of
// a team read the kv-head tiles of the same blocks at the same time (one
// block's tiles are contiguous in HBM). A wave walks its range as up to a few
// segments (one per sequence it touches): a segment that covers the whole
// sequence writes the final output; otherwise it leaves a fragment (max, sum,
// partial output) in slot 2w (the wave's first segment) or 2w+1 (its last),
// and paged_streamk_reduce_kernel combines the fragments of each split item.
// ---------------------------------------------------------------------------
constexpr int kStreamMaxSeqs = 4096;  // LDS prefix table bound
constexpr int kFragHead = 32;         // floats before a fragment's partial output (16-byte aligned)
constexpr int kStreamWaves = 4;       // waves per workgroup
// Waves per SIMD the kernel's registers must allow: the grid is sized so
// every wave is resident at once (4 SIMDs per CU).
constexpr int kStreamWavesPerSimd = 3;

struct StreamArgs {
    f16* out;
    const f16* q;
    const f16* kc;
    const f16* vc;
    const int* bt;
    const int* ctx;
    float* frag;  // [2W][kFragHead + gstride * D]: max[16], sum[16], out[gstride][D]
    // [W][4] + 1: first block of the sequence, sequence, blocks of the
    // sequence (first segment of each wave, -1 if whole), then blocks per
    // team. 64-bit on purpose: no store of the kernel has the block table's
    // type.
    long long* meta;
    float scale_log2;
    int S, H, Hkv, G, nhc, MB, num_blocks;
    int W;  // waves in the grid
};

// Blocks per sequence -> exclusive prefix in s_pre[0..S] (s_pre[S] = total),
// clamped context lengths in s_len. All threads of the workgroup take part.
// A: any argument struct with S, ctx and MB.
// Returns the longest length; s_most: one entry per wave. Up to 64 sequences are
// scanned in registers, a lane each, with one barrier.
template <typename A>
__device__ __forceinline__ int stream_prefix(const A& a, int* s_pre, int* s_len, int* s_tot, int* s_most) {
    if (a.S <= 64) {
        const int c = threadIdx.x & 63;
        const int L0 = c < a.S ? max(a.ctx[c], 0) : 0;
        const int nb = min((L0 + kBlockTokens - 1) / kBlockTokens, a.MB);
        const int len = min(L0, nb * kBlockTokens);
        const int incl = wave_inclusive_scan(nb);
        if (threadIdx.x < 64 && c < a.S) {
            s_len[c] = len;
            s_pre[c] = incl - nb;
            if (c == a.S - 1) s_pre[a.S] = incl;
        }
        __syncthreads();
        return wave_max(len);
    }
    const int chunk = (a.S + blockDim.x - 1) / blockDim.x;
    const int c0 = threadIdx.x * chunk;
    int run = 0;
    int most = 0;
    for (int c = c0; c < min(a.S, c0 + chunk); ++c) {
        const int L0 = max(a.ctx[c], 0);
        const int nb = min((L0 + kBlockTokens - 1) / kBlockTokens, a.MB);
        s_len[c] = min(L0, nb * kBlockTokens);
        most = max(most, min(L0, nb * kBlockTokens));
        s_pre[c] = run;  // local exclusive prefix, offset added below
        run += nb;
    }
    s_tot[threadIdx.x] = run;
    most = wave_max(most);
    if ((threadIdx.x & 63) == 0) s_most[threadIdx.x >> 6] = most;
    __syncthreads();
    if (threadIdx.x < 64) {
        // exclusive scan of the (<= 256) chunk totals by wave 0
        const int n = blockDim.x;
        int v[4];
        int sum = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = threadIdx.x * 4 + i;
            v[i] = idx < n ? s_tot[idx] : 0;
            sum += v[i];
        }
        const int incl = wave_inclusive_scan(sum);
        int ex = incl - sum;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = threadIdx.x * 4 + i;
            if (idx < n) s_tot[idx] = ex;
            ex += v[i];
        }
        if (threadIdx.x == 63) s_pre[a.S] = incl;
    }
    __syncthreads();
    const int off = s_tot[threadIdx.x];
    for (int c = c0; c < min(a.S, c0 + chunk); ++c) s_pre[c] += off;
    for (int w = 0; w < static_cast<int>(blockDim.x) / 64; ++w) most = max(most, s_most[w]);
    __syncthreads();
    return most;
}

template <int D>
__global__ __launch_bounds__(64 * kStreamWaves) __attribute__((amdgpu_waves_per_eu(kStreamWavesPerSimd)))
void paged_decode_streamk_kernel(const StreamArgs a) {
    constexpr int NJ = D / 16;
    extern __shared__ int s_dyn[];
    int* s_pre = s_dyn;              // [S + 1]
    int* s_len = s_dyn + a.S + 1;    // [S]
    __shared__ int s_tot[64 * kStreamWaves];
    __shared__ int s_most[kStreamWaves];
    stream_prefix(a, s_pre, s_len, s_tot, s_most);

    // Sequences without blocks are not in the list: zero their outputs here.
    for (int sz = blockIdx.x; sz < a.S; sz += gridDim.x) {
        if (s_pre[sz + 1] == s_pre[sz]) {
            for (int i = threadIdx.x; i < a.H * D; i += blockDim.x) {
                a.out[static_cast<size_t>(sz) * a.H * D + i] = static_cast<f16>(0.0f);
            }
        }
    }

    const int lane = threadIdx.x & 63;
    const int w = blockIdx.x * kStreamWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15;
    const int kg = lane >> 4;
    const int gstride = min(16, a.G);
    const int TS = a.Hkv * a.nhc;  // waves per team
    const int teams = a.W / TS;
    const int team = w / TS;
    const int member = w - team * TS;
    const int kvh = member / a.nhc;
    const int hc = member - kvh * a.nhc;
    const int g0 = hc * 16;
    const int gn = min(16, a.G - g0);
    const int h0 = kvh * a.G + g0;
    const int U = __builtin_amdgcn_readfirstlane(s_pre[a.S]);
    const int q = (U + teams - 1) / teams;
    const int u0 = team < teams ? min(U, team * q) : U;
    const int u1 = team < teams ? min(U, u0 + q) : U;
    long long* meta = a.meta + 4 * w;
    if (lane == 0) meta[0] = -1;  // no split first segment (overwritten below if there is one)
    if (w == 0 && lane == 0) a.meta[4 * a.W] = q;  // blocks per team, for the reduce

    h4 ident;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        ident[i] = (4 * kg + i == r) ? static_cast<f16>(1.0f) : static_cast<f16>(0.0f);
    }
    const int loff = kv_elem_offset(r, 4 * kg);

    bool first_seg = true;
    int u = u0;
    while (u < u1) {
        // sequence of block u: largest s with s_pre[s] <= u
        int lo = 0, hi = a.S;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (s_pre[mid] <= u) lo = mid; else hi = mid;
        }
        // Everything below is wave-uniform; readfirstlane keeps it in scalar
        // registers so the block-table reads stay scalar loads.
        const int s = __builtin_amdgcn_readfirstlane(lo);
        const int L = __builtin_amdgcn_readfirstlane(s_len[s]);
        const int pre = __builtin_amdgcn_readfirstlane(s_pre[s]);
        const int nb = __builtin_amdgcn_readfirstlane(s_pre[s + 1]) - pre;
        const int j0 = u - pre;
        const int seg = min(nb - j0, u1 - u);

        QOperand<D> qB;
        {
            const f16* qp = a.q + (static_cast<size_t>(s) * a.H + h0 + min(r, gn - 1)) * D + 4 * kg;
#pragma unroll
            for (int J = 0; J < NJ; ++J) {
                const h4 v = *reinterpret_cast<const h4*>(qp + 16 * J);
                qB.v[J] = (r < gn) ? v : h4{0, 0, 0, 0};
            }
        }
        const const_int* btrow = as_const(a.bt) + static_cast<size_t>(s) * a.MB;
        WaveState<D> st;
        st.m = -INFINITY;
        st.l = 0.0f;
#pragma unroll
        for (int J = 0; J < NJ; ++J) st.acc[J] = f4{0, 0, 0, 0};
        attend_blocks<D>(st, btrow, j0, 1, seg, L, a.kc, a.vc, a.Hkv, a.num_blocks, kvh, loff, kg,
                         qB, ident, a.scale_log2);
        float l_run = st.l;
        l_run = sum_over_kg(l_run);
        const float inv = (l_run > 0.0f) ? 1.0f / l_run : 0.0f;
        if (j0 == 0 && seg == nb) {
            if (r < gn) {
                f16* op = a.out + (static_cast<size_t>(s) * a.H + h0 + r) * D + 4 * kg;
#pragma unroll
                for (int J = 0; J < NJ; ++J) {
                    h4 o;
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] = static_cast<f16>(st.acc[J][i] * inv);
                    *reinterpret_cast<h4*>(op + 16 * J) = o;
                }
            }
        } else {
            const int slot = 2 * w + (first_seg ? 0 : 1);
            float* f = a.frag + static_cast<size_t>(slot) * (kFragHead + gstride * D);
            if (r < gn) {
                if (kg == 0) {
                    f[r] = st.m;
                    f[16 + r] = l_run;
                }
                float* fo = f + kFragHead + static_cast<size_t>(r) * D + 4 * kg;
#pragma unroll
                for (int J = 0; J < NJ; ++J) *reinterpret_cast<f4*>(fo + 16 * J) = st.acc[J] * inv;
            }
            if (first_seg && lane == 0) {
                meta[0] = pre;  // first block of the sequence in the list
                meta[1] = s;
                meta[2] = nb;
            }
        }
        first_seg = false;
        u += seg;
    }
}

// Combines the fragments of every split item: one wave per (w, g) reduces
// query head g of the item whose fragments wave w owns (four heads per
// workgroup). Wave w owns the item of its
// first segment when that segment is split, starts inside the sequence, and
// w's team is the first team to start inside it (every other workgroup exits
// at once). Fragments of the item come from the waves with the same team
// member index in teams ta..tb.
struct StreamReduceArgs {
    f16* out;
    const float* frag;
    const long long* meta;
    int H, Hkv, G, nhc, W;
    int gstride;
};

template <int D>
__global__ __launch_bounds__(256) void paged_streamk_reduce_kernel(const StreamReduceArgs a) {
    const int w = blockIdx.x;
    const int g = blockIdx.y * 4 + (threadIdx.x >> 6);
    const long long* m = a.meta + 4 * w;
    if (m[0] < 0) return;
    const int TS = a.Hkv * a.nhc;
    const int q = static_cast<int>(a.meta[4 * a.W]);
    const int ustart = static_cast<int>(m[0]);
    const int team = w / TS;
    const int ta = ustart / q;
    if (team != ta + 1 || ustart == team * q) return;  // not the owner
    const int member = w - team * TS;
    const int kvh = member / a.nhc;
    const int hc = member - kvh * a.nhc;
    const int g0 = hc * 16;
    const int gn = min(16, a.G - g0);
    if (g >= gn) return;
    const int s = static_cast<int>(m[1]);
    const int nb = static_cast<int>(m[2]);
    const int P = (ustart + nb - 1) / q - ta + 1;
    const size_t fs = kFragHead + static_cast<size_t>(a.gstride) * D;
    // fragment i of the item comes from team ta + i
    auto frag_of = [&](int i) {
        const int t = ta + i;
        const int v = t * TS + member;
        const int slot = (t == ta && ta * q < ustart) ? 2 * v + 1 : 2 * v;
        return a.frag + slot * fs;
    };
    f16* o = a.out + (static_cast<size_t>(s) * a.H + kvh * a.G + g0 + g) * D;
    combine_head_wave<D>(
        P, [&](int i) { return frag_of(i)[g]; }, [&](int i) { return frag_of(i)[16 + g]; },
        [&](int i) { return frag_of(i) + kFragHead + static_cast<size_t>(g) * D; },
        [&](int d, float v) { o[d] = static_cast<f16>(v); });
}

// ---------------------------------------------------------------------------
// Split-K by teams, for batches of few sequences. The blocks of all sequences
// form one list, as in the balanced mode, but a team is TS = Hkv * nhc
// workgroups (one per kv head and head chunk) instead of waves: team t takes
// blocks [t*q, (t+1)*q), q = ceil(blocks / teams), and the four waves of a
// workgroup take a range's blocks round-robin and merge through LDS. Every
// workgroup gets the same number of blocks whatever the context lengths, and
// a head is left with one fragment per team that touches its sequence, at
// most teams + 1 per sequence, whatever partition size the caller asks for.
// A range that covers a whole sequence writes its output; otherwise its first
// segment leaves a fragment in the workgroup's even slot and its last one in
// the odd slot, and paged_team_reduce_kernel combines them. Where all contexts
// are short (team_whole_blocks) the teams take whole sequences instead, one
// after the other (blocks per team 0: the reduce has nothing to do); the table's
// width does not tell, so the kernel looks at the lengths.
//
// Bound: HBM for long contexts, for short ones the latency of two dependent
// kernels. Measured on MI355X (us per call, 512-token partitions; before: a
// range per wave, cut at partition ends, so a head of one sequence had 256
// fragments): 1 sequence of 7919 tokens, 32/8 heads x 128, 25.1 -> 12.8; of
// 32768 39.3 -> 27.3; 4000 tokens, 64/8 heads 49.0 -> 12.4; 8 x 32768 tokens,
// 64/8 heads 170.5 -> 164.5 (16.8 MB of partials became 2 MB); 64 x
// 512-4096 102.7 -> 97.1. Two workgroups per CU: three (168 registers) took
// 14.8, 28.6, 14.0, 168.4 and 98.7 on those; one of eight waves 12.8, 27.3,
// 11.7, 162.9 and 97.5, but 35.3 against 32.1 on 64 lognormal contexts of 8
// heads x 64 and 54.6 against 50.4 on 32 of 16 x 128, where a segment is
// short and its waves run dry.
// ---------------------------------------------------------------------------
constexpr int kTeamWaves = 4;
constexpr int kTeamPerCU = 2;  // workgroups per CU: two waves per SIMD

// Blocks of the longest context up to which teams take whole sequences. Cut, a
// context of few sequences spreads over the teams it would leave idle, so the
// line rises with the sequences per team. Measured with tables 512 blocks wide
// (us per call, cut / whole, 32/8 heads x 128, 64 teams): 1 sequence of 128
// tokens 7.7 / 7.2, 192 7.7 / 7.6, 256 7.7 / 8.1; 4 of 256 8.7 / 8.1, 384 8.7 /
// 9.2; 16 of 384 11.2 / 10.1, 512 11.9 / 11.7; 64 of 16-512 24.7 / 17.5; 96 of
// 16-128 19.8 / 11.7.
__device__ __forceinline__ int team_whole_blocks(int S, int teams) {
    return min((12 + 64 * S / teams) & ~3, 32);
}

struct TeamArgs {
    f16* out;
    const f16* q;
    const f16* kc;
    const f16* vc;
    const int* bt;
    const int* ctx;
    float* frag;  // [2 * teams * TS][kFragHead + gstride * D]
    int* meta;    // for the reduce: [0] blocks per team (0: nothing was cut), [1 .. S + 1] block prefix
    float scale_log2;
    int S, H, Hkv, G, nhc, MB, num_blocks;
    int teams;
};

template <int D>
__global__ __launch_bounds__(64 * kTeamWaves) __attribute__((amdgpu_waves_per_eu(kTeamPerCU)))
void paged_team_kernel(const TeamArgs a) {
    constexpr int NJ = D / 16;
    constexpr int NW = kTeamWaves;
    extern __shared__ __align__(16) float smem[];
    const int gstride = min(16, a.G);
    int* s_pre = reinterpret_cast<int*>(smem + merge_lds_floats<D, NW>(a.G));  // [S + 1]
    int* s_len = s_pre + a.S + 1;                                              // [S]
    __shared__ int s_tot[64 * NW];
    __shared__ int s_most[NW];
    const int most = stream_prefix(a, s_pre, s_len, s_tot, s_most);

    const int U = __builtin_amdgcn_readfirstlane(s_pre[a.S]);
    const bool whole = __builtin_amdgcn_readfirstlane(most) <= team_whole_blocks(a.S, a.teams) * kBlockTokens;
    const int q = whole ? 0 : (U + a.teams - 1) / a.teams;
    if (blockIdx.x == 0) {
        for (int i = threadIdx.x; i <= a.S; i += blockDim.x) a.meta[1 + i] = s_pre[i];
        if (threadIdx.x == 0) a.meta[0] = q;
    }
    // Sequences without blocks are not in the list: zero their outputs here.
    for (int sz = blockIdx.x; sz < a.S; sz += gridDim.x) {
        if (s_pre[sz + 1] == s_pre[sz]) {
            for (int i = threadIdx.x; i < a.H * D; i += blockDim.x) {
                a.out[static_cast<size_t>(sz) * a.H * D + i] = static_cast<f16>(0.0f);
            }
        }
    }
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15;
    const int kg = lane >> 4;
    const int TS = a.Hkv * a.nhc;
    const int team = blockIdx.x / TS;
    const int member = blockIdx.x - team * TS;
    const int kvh = member / a.nhc;
    const int hc = member - kvh * a.nhc;
    const int g0 = hc * 16;
    const int gn = min(16, a.G - g0);
    const int h0 = kvh * a.G + g0;
    const int u0 = min(U, team * q);
    const int u1 = min(U, u0 + q);

    h4 ident;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        ident[i] = (4 * kg + i == r) ? static_cast<f16>(1.0f) : static_cast<f16>(0.0f);
    }
    const int loff = kv_elem_offset(r, 4 * kg);
    int u = u0;           // whole: unused
    int next = team;      // whole: the team's next sequence
    bool first = true;    // the workgroup's first segment
    while (whole ? next < a.S : u < u1) {
        int lo = next, hi = a.S;
        if (whole) {
            next += a.teams;
            if (s_pre[lo + 1] == s_pre[lo]) continue;
        } else {
            lo = 0;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (s_pre[mid] <= u) lo = mid; else hi = mid;
            }
        }
        // Wave-uniform, in scalar registers, so the block-table reads stay
        // scalar loads.
        const int s = __builtin_amdgcn_readfirstlane(lo);
        const int L = __builtin_amdgcn_readfirstlane(s_len[s]);
        const int pre = __builtin_amdgcn_readfirstlane(s_pre[s]);
        const int nb = __builtin_amdgcn_readfirstlane(s_pre[s + 1]) - pre;
        const int j0 = whole ? 0 : u - pre;
        const int seg = whole ? nb : min(nb - j0, u1 - u);
        QOperand<D> qB;
        {
            const f16* qp = a.q + (static_cast<size_t>(s) * a.H + h0 + min(r, gn - 1)) * D + 4 * kg;
#pragma unroll
            for (int J = 0; J < NJ; ++J) {
                const h4 v = *reinterpret_cast<const h4*>(qp + 16 * J);
                qB.v[J] = (r < gn) ? v : h4{0, 0, 0, 0};
            }
        }
        const const_int* btrow = as_const(a.bt) + static_cast<size_t>(s) * a.MB;
        WaveState<D> st;
        st.m = -INFINITY;
        st.l = 0.0f;
#pragma unroll
        for (int J = 0; J < NJ; ++J) st.acc[J] = f4{0, 0, 0, 0};
        attend_blocks<D>(st, btrow, j0 + w, NW, (seg - w + NW - 1) / NW, L, a.kc, a.vc, a.Hkv,
                         a.num_blocks, kvh, loff, kg, qB, ident, a.scale_log2);
        const float l_run = sum_over_kg(st.l);
        const bool direct = j0 == 0 && seg == nb;
        float* f = a.frag + static_cast<size_t>(2 * blockIdx.x + !first) * (kFragHead + gstride * D);
        if (!first) __syncthreads();  // the segment before has been read from LDS
        first = false;
        merge_waves<D, NW>(smem, st, l_run, gn, gstride, w, r, kg, [&](int g, int d, float o, float M, float den) {
            if (direct) {
                a.out[(static_cast<size_t>(s) * a.H + h0 + g) * D + d] = static_cast<f16>(o);
            } else {
                f[kFragHead + g * D + d] = o;
                if (d == 0) {
                    f[g] = M;
                    f[16 + g] = den;
                }
            }
        });
        u += seg;
    }
}

// One (query head, sequence) per workgroup: its fragments come from the teams
// whose ranges touch the sequence. A fragment is its team's first segment
// (even slot) unless the sequence starts inside that team's range.
struct TeamReduceArgs {
    f16* out;
    const float* frag;
    const int* meta;
    int H, G, nhc, TS, gstride;
};

template <int D>
__global__ __launch_bounds__(256) void paged_team_reduce_kernel(const TeamReduceArgs a) {
    const int s = blockIdx.y;
    const int h = blockIdx.x;
    const int q = a.meta[0];
    const int pre = a.meta[1 + s];
    const int nb = a.meta[2 + s] - pre;
    if (nb == 0 || q == 0) return;
    const int ta = pre / q;
    const int P = (pre + nb - 1) / q - ta + 1;
    if (P == 1) return;  // written by its team
    const int kvh = h / a.G;
    const int gk = h - kvh * a.G;
    const int hc = gk / 16;
    const int g = gk - hc * 16;
    const int member = kvh * a.nhc + hc;
    const size_t fs = kFragHead + static_cast<size_t>(a.gstride) * D;
    const bool late = pre > ta * q;  // the sequence starts inside its first team's range
    auto frag_of = [&](int i) {
        return a.frag + static_cast<size_t>(2 * ((ta + i) * a.TS + member) + (i == 0 && late)) * fs;
    };
    f16* o = a.out + (static_cast<size_t>(s) * a.H + h) * D;
    combine_head_split<D, 4>(
        P, [&](int i) { return frag_of(i)[g]; }, [&](int i) { return frag_of(i)[16 + g]; },
        [&](int i) { return frag_of(i) + kFragHead + static_cast<size_t>(g) * D; },
        [&](int d, float v) { o[d] = static_cast<f16>(v); });
}

// Bit-exact materialisation of one (sequence, kv head) through the tile
// addressing above.
struct GatherArgs {
    const uint16_t* kc;
    const uint16_t* vc;
    const int* bt;
    const int* ctx;
    uint16_t* ko;
    uint16_t* vo;
    int s, kvh, Hkv, D, MB, max_len;
};

__global__ __launch_bounds__(256) void gather_kv_kernel(const GatherArgs a) {
    int L = max(a.ctx[a.s], 0);
    L = min(L, min(a.MB * kBlockTokens, a.max_len));
    const int* btrow = a.bt + static_cast<size_t>(a.s) * a.MB;
    const size_t n = static_cast<size_t>(a.max_len) * a.D;
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const int t = static_cast<int>(i / a.D);
        const int d = static_cast<int>(i - static_cast<size_t>(t) * a.D);
        uint16_t kv = 0, vv = 0;
        if (t < L) {
            const int b = btrow[t / kBlockTokens];
            const size_t off = kv_tile_offset(b, a.kvh, a.Hkv, a.D) + kv_elem_offset(d, t % kBlockTokens);
            kv = a.kc[off];
            vv = a.vc[off];
        }
        a.ko[i] = kv;
        a.vo[i] = vv;
    }
}

struct ClearArgs {
    uint32_t* p;
    size_t words;
};

__global__ __launch_bounds__(256) void clear_kernel(const ClearArgs a) {
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < a.words;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        a.p[i] = 0u;
    }
}


// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
constexpr size_t kAlign = 256;

size_t align_up(size_t x) { return (x + kAlign - 1) / kAlign * kAlign; }

struct Shape {
    int S, H, Hkv, D, BS, MB;
};

int validate_decode(const char* who, const void* out, const void* q, const void* kc,
                    const void* vc, const int* bt, const int* ctx, const Shape& sh) {
    if (sh.S < 0 || sh.H <= 0 || sh.Hkv <= 0 || sh.MB < 0) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER,
                    "%s: num_seqs=%d num_heads=%d num_kv_heads=%d max_num_blocks_per_seq=%d",
                    who, sh.S, sh.H, sh.Hkv, sh.MB);
    }
    if (sh.H % sh.Hkv != 0) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER,
                    "%s: num_heads %d is not a multiple of num_kv_heads %d", who, sh.H, sh.Hkv);
    }
    if (sh.D != 64 && sh.D != 128) {
        return fail(SWIFTLLM_ERR_NOT_SUPPORTED, "%s: head_dim %d (supported: 64, 128)", who, sh.D);
    }
    if (sh.BS != kBlockTokens) {
        return fail(SWIFTLLM_ERR_NOT_SUPPORTED, "%s: block_size %d (supported: 16)", who, sh.BS);
    }
    if (sh.S > 65535) {
        return fail(SWIFTLLM_ERR_NOT_SUPPORTED, "%s: num_seqs %d > 65535", who, sh.S);
    }
    const long long nhc = (sh.H / sh.Hkv + 15) / 16;
    if (static_cast<long long>(sh.Hkv) * nhc > 65535) {
        return fail(SWIFTLLM_ERR_NOT_SUPPORTED, "%s: too many kv heads", who);
    }
    if (sh.S == 0) return SWIFTLLM_OK;
    if (!out || !q || !kc || !vc || !bt || !ctx) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: null pointer", who);
    }
    if (!aligned(out, 2) || !aligned(q, 8) || !aligned(kc, 8) || !aligned(vc, 8) ||
        !aligned(bt, 4) || !aligned(ctx, 4)) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER,
                    "%s: misaligned pointer (query and caches need 8-byte alignment)", who);
    }
    return SWIFTLLM_OK;
}

// Waves per workgroup of the single-pass kernel: the whole context of a
// (sequence, kv head) is one workgroup, so it gets the most waves.
#ifndef SWIFTLLM_WAVES_V1
#define SWIFTLLM_WAVES_V1 4
#endif
constexpr int kWavesV1 = SWIFTLLM_WAVES_V1;
constexpr int kWavesV1Wide = 8;
// Blocks per sequence up to which several rounds of single-pass workgroups
// run in plain order.
constexpr int kSingleRoundBlocks = 64;
constexpr int kListMaxSeqs = 512;
// Waves per workgroup of a split-K partition.
#ifndef SWIFTLLM_WAVES_V2
#define SWIFTLLM_WAVES_V2 4
#endif
constexpr int kWavesV2 = SWIFTLLM_WAVES_V2;

template <int D, int NW>
hipError_t launch_decode_t(const DecodeArgs& a, hipStream_t stream) {
    const size_t lds = static_cast<size_t>(merge_lds_floats<D, NW>(a.G)) * sizeof(float);
    const dim3 grid(1, a.Hkv * a.nhc, a.S);
    return launch(paged_decode_kernel<D, NW>, grid, dim3(NW * 64), lds, stream, a);
}

template <int NW>
hipError_t launch_decode(const DecodeArgs& a, int D, hipStream_t stream) {
    return D == 128 ? launch_decode_t<128, NW>(a, stream) : launch_decode_t<64, NW>(a, stream);
}

template <int D, int NW>
hipError_t launch_partition_t(const DecodeArgs& a, unsigned grid, hipStream_t stream) {
    size_t lds = static_cast<size_t>(merge_lds_floats<D, NW>(a.G)) * sizeof(float);
    if (a.S <= kPartMaxSeqs) lds += part_list_lds_bytes(a.S);
    return launch(paged_partition_kernel<D, NW>, dim3(grid), dim3(NW * 64), lds, stream, a);
}

int device_cus();

// kItemShare of what one of the partition kernel's resident workgroups (three
// per CU) gets of a batch, per block of it.
float item_share(const DecodeArgs& a) {
    return kItemShare * static_cast<float>(a.Hkv * a.nhc) / static_cast<float>(3 * device_cus());
}

// Split-K partition kernel: a grid of resident workgroups (three 4-wave
// workgroups per CU, four rounds) walking the compacted item list, or one
// workgroup per possible item for batches too large to compact in LDS.
template <int NW>
hipError_t launch_partition(const DecodeArgs& a, int D, hipStream_t stream, bool* too_large) {
    const long long possible = static_cast<long long>(a.MP) * a.Hkv * a.nhc * a.S;
    long long grid = possible;
    if (a.S <= kPartMaxSeqs) grid = std::min(possible, 12LL * device_cus());
    *too_large = grid > 0x7fffffffLL;
    if (*too_large || grid <= 0) return hipSuccess;
    const unsigned g = static_cast<unsigned>(grid);
    return D == 128 ? launch_partition_t<128, NW>(a, g, stream)
                    : launch_partition_t<64, NW>(a, g, stream);
}

DecodeArgs make_args(void* out, const void* q, const void* kc, const void* vc, const int* bt,
                     const int* ctx, float scale, const Shape& sh, int num_blocks) {
    DecodeArgs a{};
    a.out = static_cast<f16*>(out);
    a.q = static_cast<const f16*>(q);
    a.kc = static_cast<const f16*>(kc);
    a.vc = static_cast<const f16*>(vc);
    a.bt = bt;
    a.ctx = ctx;
    a.scale_log2 = static_cast<float>(static_cast<double>(scale) * static_cast<double>(kLog2e));
    a.H = sh.H;
    a.Hkv = sh.Hkv;
    a.G = sh.H / sh.Hkv;
    a.nhc = (a.G + 15) / 16;
    a.MB = sh.MB;
    a.S = sh.S;
    a.num_blocks = num_blocks;
    return a;
}


int decode_v1(void* out, const void* q, const void* kc, const void* vc, const int* bt,
              const int* ctx, float scale, const Shape& sh, int num_blocks, hipStream_t stream,
              const char* who) {
    int rc = validate_decode(who, out, q, kc, vc, bt, ctx, sh);
    if (rc != SWIFTLLM_OK) return rc;
    if ((rc = require_device()) != SWIFTLLM_OK) return rc;
    if (sh.S == 0) return ok();
    DecodeArgs a = make_args(out, q, kc, vc, bt, ctx, scale, sh, num_blocks);
    a.part_blocks = 0;
    a.MP = 1;
    const int cus = device_cus();
    const long long items = static_cast<long long>(sh.S) * a.Hkv * a.nhc;
    // At most one workgroup per CU: eight waves each, so a context is half as
    // long a chain (16 query heads would need more LDS for the merge).
    // Measured (us per call, 4 waves -> 8): 1 x 1024 tokens of 32/8 heads x 128
    // 12.5 -> 11.4, 32 x 512 13.9 -> 12.4, 4 x 2048 of 8 heads x 64 16.5 ->
    // 13.7. At 64 x 32-512 (512 items) 15.8 -> 18.5, so not beyond.
    if (items <= cus && a.G <= 8) {
        return launched(launch_decode<kWavesV1Wide>(a, sh.D, stream), who);
    }
    if (items <= 3LL * cus) {
        // The whole grid is resident at once (three 4-wave workgroups per CU
        // at the kernel's register count): snake order over the ranked
        // sequences when there are few enough to rank.
        a.snake = sh.S <= kLptMaxSeqs ? cus : 0;
    } else if (sh.MB > kSingleRoundBlocks && sh.S <= kListMaxSeqs) {
        // Several rounds of workgroups, and tables that may hold contexts long
        // enough for the last ones to leave a tail: the partition kernel, one
        // item per sequence and kv head, which takes them longest first where
        // that pays (list_pays). Of more sequences the list costs more than a
        // tail of theirs: 600, one of 2500 tokens and the others 32, 48.8 in
        // plain order, 55.8 by the list.
        a.single = true;
        a.part_blocks = std::min(sh.MB, 1 << 27);  // 2^31 tokens
        a.share = item_share(a);
        bool too_large = false;
        return launched(launch_partition<kWavesV2>(a, sh.D, stream, &too_large), who);
    }
    return launched(launch_decode<kWavesV1>(a, sh.D, stream), who);
}

// Whether a split-K call runs single pass instead: its tables are too short
// for a split to pay for the second kernel. The longest context is at most MB
// blocks; a single pass takes about 5 us + 0.08-0.165 us per block of it, a
// split 7.5-9.5 us at least, and with items enough for every CU the single
// pass reads at the same rate. Measured (us per call, single pass / teams,
// all contexts of one length, 32/8 heads x 128): 1 sequence of 512 tokens 7.8
// / 8.2, of 1024 11.4 / 9.1; 8 of 512 9.2 / 10.8, of 1024 14.9 / 12.8; 16 of
// 1024 16.4 / 17.4; 64 of 64-1024 25.9 / 34.1; items: 128 of 200-400 28.8 /
// 31.0, 256 of 1-1024 lognormal 106 / 105.
// The table says nothing of the other contexts, and one long context among
// short ones is the single pass's worst: its whole chain runs on one workgroup
// per kv head. So a table past 96 blocks is split whatever the batch, and past
// 64 (32 with more than four items per CU) in balanced mode, whose ranges are
// for such batches. All but one of 32 tokens (us per call, single pass / split):
// 64 sequences, one of 1536 tokens 22 / 26 in 512-token items (12 by teams),
// 2500 31.9 / 15.0; 96, one of 3500 43.6 / 19.1; balanced 48, one of 1280 17.0
// / 11.5, of 2048 24.3 / 11.8; 256, one of 1024 20.9 / 15.3. Even contexts pay
// for it above the line: 32 of 1536 tokens balanced 30.7 / 35.9, 64 of 128-2048
// in 512-token partitions 49.5 / 55.8, 256 of 1024 balanced 157 / 185.
bool single_pass(const Shape& sh, int partition_size, int cus) {
    if (sh.S > kPartMaxSeqs) return false;
    const bool balanced = partition_size == 0;
    const long long items = static_cast<long long>(sh.S) * sh.Hkv * ((sh.H / sh.Hkv + 15) / 16);
    if (items > 3LL * cus) return sh.MB <= (balanced && items > 4LL * cus ? 32 : 64);
    return sh.MB <= std::min(32 + items / 4, balanced ? 64LL : 96LL);
}

// Split-K workspace: max logits and exp sums [S][H][MP] and partial outputs
// [S][H][MP][D], all fp32, or the teams' fragments and their metadata. Plain
// scratch: every value a call reads was written earlier in the same call, so
// it needs no initialisation.
struct V2Need {
    int MP;          // partitions per sequence
    size_t stat;     // bytes of one [S][H][MP] float array
    size_t total;    // bytes of the whole workspace
};

V2Need v2_need(const Shape& sh, int partition_size, int cus) {
    V2Need n{};
    const int part_blocks = partition_size / kBlockTokens;
    n.MP = sh.MB == 0 ? 1 : (sh.MB + part_blocks - 1) / part_blocks;
    n.stat = align_up(sizeof(float) * static_cast<size_t>(sh.S) * sh.H * n.MP);
    n.total = 2 * n.stat + align_up(sizeof(float) * static_cast<size_t>(sh.S) * sh.H * n.MP * sh.D);
    // Few sequences and short partitions: room for eight fragments per CU and
    // the block prefix beside the partials. The teams need half of it; the
    // size is part of what callers have stored and stays.
    const int G = sh.H / sh.Hkv;
    const long long TS = static_cast<long long>(sh.Hkv) * ((G + 15) / 16);
    const long long W = 8LL * cus;
    const long long teams = TS > 0 ? W / TS : 0;
    if (sh.S <= kStreamMaxSeqs && part_blocks <= 64 && TS > 0 && TS <= W && 4LL * sh.S <= teams &&
        64LL * n.MP * sh.D < (1LL << 31)) {
        const size_t gstride = static_cast<size_t>(std::min(16, G));
        n.total += align_up(sizeof(float) * static_cast<size_t>(W) * (kFragHead + gstride * sh.D)) +
                   align_up(sizeof(int) * (static_cast<size_t>(sh.S) + 3));
    }
    return n;
}

// The team kernel's grid and workspace; teams == 0 where it does not serve
// the shape: fewer than four teams, or more than two sequences per team,
// which then have items enough for the GPU and longer ranges of their own.
// Measured (us per call, 32/8 heads x 128, contexts lognormal around 600):
// 100 sequences 87.6 by teams, 89.8 in items of 512-token partitions; 256
// 191.9 by teams, 179 in items (below).
struct TeamNeed {
    int teams, TS;
    size_t meta;   // offset of the metadata behind the fragments
    size_t total;
};

TeamNeed team_need(const Shape& sh, int cus) {
    TeamNeed n{};
    const int G = sh.H / sh.Hkv;
    const long long TS = static_cast<long long>(sh.Hkv) * ((G + 15) / 16);
    const long long teams = static_cast<long long>(cus) * kTeamPerCU / TS;
    if (teams < 4 || sh.S > 2 * teams || sh.S > kStreamMaxSeqs) return n;
    n.teams = static_cast<int>(teams);
    n.TS = static_cast<int>(TS);
    n.meta = align_up(sizeof(float) * 2 * static_cast<size_t>(teams * TS) *
                      (kFragHead + static_cast<size_t>(std::min(16, G)) * sh.D));
    n.total = n.meta + sizeof(int) * (static_cast<size_t>(sh.S) + 2);
    return n;
}

// A wave combines a head in one batch of kReduceRows rows for up to that many
// partitions per sequence; beyond, the four waves of a workgroup do.
template <int D>
hipError_t launch_reduce_t(const ReduceArgs& r, int S, hipStream_t stream) {
    if (r.MP <= kReduceRows) {
        return launch(paged_reduce_wave_kernel<D>, dim3((r.H + 3) / 4, S), dim3(256), 0, stream, r);
    }
    return launch(paged_reduce_split_kernel<D>, dim3(r.H, S), dim3(256), 0, stream, r);
}

int validate_partition(const char* who, int partition_size) {
    if (partition_size < 0 || partition_size % kBlockTokens != 0) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER,
                    "%s: partition_size %d must be 0 (balanced) or a positive multiple of 16", who,
                    partition_size);
    }
    return SWIFTLLM_OK;
}

// Balanced mode: waves resident per CU (3 per SIMD at the kernel's register
// count) times the device's CUs, so the whole grid runs in one round.
constexpr int kStreamWavesPerCU = 4 * kStreamWavesPerSimd;
constexpr int kDefaultCUs = 304;  // used to size workspaces when no device is visible

int device_cus() {
    static int cache[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return kDefaultCUs;
    if (cache[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
            return kDefaultCUs;
        }
        cache[dev] = n;
    }
    return cache[dev];
}

struct StreamNeed {
    int W;
    size_t frag, total;
};

StreamNeed stream_need(const Shape& sh, int cus) {
    StreamNeed n{};
    n.W = cus * kStreamWavesPerCU;
    const size_t gstride = static_cast<size_t>(std::min(16, sh.H / sh.Hkv));
    n.frag = align_up(sizeof(float) * 2 * static_cast<size_t>(n.W) * (kFragHead + gstride * sh.D));
    n.total = n.frag + align_up(sizeof(long long) * (4 * static_cast<size_t>(n.W) + 1));
    return n;
}

int decode_balanced(void* out, void* ws, const StreamNeed& need, const void* q, const void* kc,
                    const void* vc, const int* bt, const int* ctx, float scale, const Shape& sh,
                    int num_blocks, hipStream_t stream, const char* who) {
    DecodeArgs d = make_args(out, q, kc, vc, bt, ctx, scale, sh, num_blocks);
    StreamArgs a{};
    a.out = d.out;
    a.q = d.q;
    a.kc = d.kc;
    a.vc = d.vc;
    a.bt = bt;
    a.ctx = ctx;
    a.frag = reinterpret_cast<float*>(ws);
    a.meta = reinterpret_cast<long long*>(static_cast<char*>(ws) + need.frag);
    a.scale_log2 = d.scale_log2;
    a.S = sh.S;
    a.H = sh.H;
    a.Hkv = sh.Hkv;
    a.G = d.G;
    a.nhc = d.nhc;
    a.MB = sh.MB;
    a.num_blocks = num_blocks;
    a.W = need.W;
    const size_t lds = sizeof(int) * (2 * static_cast<size_t>(sh.S) + 1);
    const dim3 grid(need.W / kStreamWaves);
    hipError_t err = sh.D == 128
        ? launch(paged_decode_streamk_kernel<128>, grid, dim3(64 * kStreamWaves), lds, stream, a)
        : launch(paged_decode_streamk_kernel<64>, grid, dim3(64 * kStreamWaves), lds, stream, a);
    if (err != hipSuccess) return launched(err, who);
    StreamReduceArgs r{};
    r.out = a.out;
    r.frag = a.frag;
    r.meta = a.meta;
    r.H = a.H;
    r.Hkv = a.Hkv;
    r.G = a.G;
    r.nhc = a.nhc;
    r.W = a.W;
    r.gstride = std::min(16, a.G);
    const dim3 rgrid(need.W, (r.gstride + 3) / 4);
    err = sh.D == 128 ? launch(paged_streamk_reduce_kernel<128>, rgrid, dim3(256), 0, stream, r)
                      : launch(paged_streamk_reduce_kernel<64>, rgrid, dim3(256), 0, stream, r);
    return launched(err, who);
}

// The partition size a v2 call runs with: balanced mode (0) needs its
// prefix table in LDS and at least 4 teams of Hkv * nhc waves; otherwise it
// falls back to partitions of 512 tokens.
int effective_partition(const Shape& sh, int partition_size, int cus) {
    if (partition_size == 0 &&
        (sh.S > kStreamMaxSeqs ||
         static_cast<long long>(sh.Hkv) * ((sh.H / sh.Hkv + 15) / 16) * 4 > cus * kStreamWavesPerCU)) {
        return 512;
    }
    return partition_size;
}

// Workspace bytes a v2 call with this (effective) partition size uses.
size_t v2_bytes(const Shape& sh, int partition_size, int cus) {
    return partition_size == 0 ? stream_need(sh, cus).total : v2_need(sh, partition_size, cus).total;
}

// The team kernel, then its reduce; ws holds need.total bytes.
int decode_team(void* out, void* ws, const void* q, const void* kc, const void* vc, const int* bt,
                const int* ctx, float scale, const Shape& sh, int num_blocks, const TeamNeed& need,
                hipStream_t stream, const char* who) {
    const DecodeArgs d = make_args(out, q, kc, vc, bt, ctx, scale, sh, num_blocks);
    TeamArgs a{};
    a.out = d.out;
    a.q = d.q;
    a.kc = d.kc;
    a.vc = d.vc;
    a.bt = bt;
    a.ctx = ctx;
    a.frag = static_cast<float*>(ws);
    a.meta = reinterpret_cast<int*>(static_cast<char*>(ws) + need.meta);
    a.scale_log2 = d.scale_log2;
    a.S = sh.S;
    a.H = sh.H;
    a.Hkv = sh.Hkv;
    a.G = d.G;
    a.nhc = d.nhc;
    a.MB = sh.MB;
    a.num_blocks = num_blocks;
    a.teams = need.teams;
    // Dynamic LDS: the wave merge, then the block prefix and the lengths.
    const size_t merge = sizeof(float) * static_cast<size_t>(sh.D == 128 ? merge_lds_floats<128, kTeamWaves>(a.G)
                                                                         : merge_lds_floats<64, kTeamWaves>(a.G));
    const size_t lds = merge + sizeof(int) * (2 * static_cast<size_t>(sh.S) + 1);
    const dim3 grid(static_cast<unsigned>(need.teams * need.TS));
    const dim3 block(64 * kTeamWaves);
    hipError_t err = sh.D == 128 ? launch(paged_team_kernel<128>, grid, block, lds, stream, a)
                                 : launch(paged_team_kernel<64>, grid, block, lds, stream, a);
    if (err != hipSuccess) return launched(err, who);
    TeamReduceArgs r{};
    r.out = a.out;
    r.frag = a.frag;
    r.meta = a.meta;
    r.H = a.H;
    r.G = a.G;
    r.nhc = a.nhc;
    r.TS = need.TS;
    r.gstride = std::min(16, a.G);
    const dim3 rgrid(a.H, sh.S);
    err = sh.D == 128 ? launch(paged_team_reduce_kernel<128>, rgrid, dim3(256), 0, stream, r)
                      : launch(paged_team_reduce_kernel<64>, rgrid, dim3(256), 0, stream, r);
    return launched(err, who);
}

int decode_v2(void* out, void* ws, size_t ws_bytes, const void* q, const void* kc, const void* vc,
              const int* bt, const int* ctx, float scale, const Shape& sh, int partition_size,
              int num_blocks, hipStream_t stream, const char* who) {
    int rc = validate_decode(who, out, q, kc, vc, bt, ctx, sh);
    if (rc != SWIFTLLM_OK) return rc;
    if ((rc = validate_partition(who, partition_size)) != SWIFTLLM_OK) return rc;
    partition_size = effective_partition(sh, partition_size, device_cus());
    if (partition_size == 0) {
        if (sh.S > 0 && (ws == nullptr || !aligned(ws, 256))) {
            return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: workspace null or not 256-byte aligned", who);
        }
        if ((rc = require_device()) != SWIFTLLM_OK) return rc;
        if (sh.S == 0) return ok();
        const StreamNeed need = stream_need(sh, device_cus());
        if (ws_bytes < need.total) {
            return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: workspace of %zu bytes, %zu needed", who,
                        ws_bytes, need.total);
        }
        if (single_pass(sh, partition_size, device_cus())) {
            return decode_v1(out, q, kc, vc, bt, ctx, scale, sh, num_blocks, stream, who);
        }
        const TeamNeed team = team_need(sh, device_cus());
        if (team.teams > 0 && team.total <= need.total) {
            return decode_team(out, ws, q, kc, vc, bt, ctx, scale, sh, num_blocks, team, stream, who);
        }
        return decode_balanced(out, ws, need, q, kc, vc, bt, ctx, scale, sh, num_blocks, stream, who);
    }
    const V2Need need = v2_need(sh, partition_size, device_cus());
    if (sh.S > 0) {
        if (ws == nullptr || !aligned(ws, 256)) {
            return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: workspace null or not 256-byte aligned", who);
        }
        if (ws_bytes < need.total) {
            return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: workspace of %zu bytes, %zu needed", who,
                        ws_bytes, need.total);
        }
    }
    if ((rc = require_device()) != SWIFTLLM_OK) return rc;
    if (sh.S == 0) return ok();
    if (single_pass(sh, partition_size, device_cus())) {
        return decode_v1(out, q, kc, vc, bt, ctx, scale, sh, num_blocks, stream, who);
    }
    const TeamNeed team = team_need(sh, device_cus());
    if (team.teams > 0 && team.total <= need.total) {
        return decode_team(out, ws, q, kc, vc, bt, ctx, scale, sh, num_blocks, team, stream, who);
    }
    DecodeArgs a = make_args(out, q, kc, vc, bt, ctx, scale, sh, num_blocks);
    char* base = static_cast<char*>(ws);
    a.ws_max = reinterpret_cast<float*>(base);
    a.ws_sum = reinterpret_cast<float*>(base + need.stat);
    a.ws_out = reinterpret_cast<float*>(base + 2 * need.stat);
    a.part_blocks = partition_size / kBlockTokens;
    a.MP = need.MP;
    a.share = item_share(a);
    bool too_large = false;
    hipError_t err = launch_partition<kWavesV2>(a, sh.D, stream, &too_large);
    if (too_large) {
        return fail(SWIFTLLM_ERR_NOT_SUPPORTED, "%s: %d sequences x %d partitions is too many",
                    who, sh.S, need.MP);
    }
    if (err != hipSuccess || need.MP <= 1) return launched(err, who);
    ReduceArgs r{};
    r.out = a.out;
    r.ctx = ctx;
    r.ws_max = a.ws_max;
    r.ws_sum = a.ws_sum;
    r.ws_out = a.ws_out;
    r.S = a.S;
    r.H = a.H;
    r.MB = a.MB;
    r.part_blocks = a.part_blocks;
    r.MP = a.MP;
    r.share = a.share;
    err = sh.D == 128 ? launch_reduce_t<128>(r, sh.S, stream)
                      : launch_reduce_t<64>(r, sh.S, stream);
    return launched(err, who);
}

}  // namespace
}  // namespace swiftllm

// ---------------------------------------------------------------------------
// Split-K decode with no allocation. Some callers cannot allocate (code under
// HIP graph capture, tight serving loops, harnesses that forbid hipMalloc),
// so swiftllm_hip_launch_paged_attention_v2_noalloc takes its workspace from
// this static device array instead of an argument. Each device that loads the
// library holds its own copy until the process ends. All calls on a device
// share that copy: calls that overlap on one device (several streams or host
// threads) race on it and must be ordered on one stream. The split-K
// workspace is plain scratch (a call reads only what it wrote first), so
// nothing is cleared between calls.
// ---------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[SWIFTLLM_HIP_NOALLOC_SCRATCH_BYTES];

namespace swiftllm {
namespace {

constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch[kMaxScratchDevices] = {};

// Device address of `scratch` on the current device, looked up on the first
// call on that device. In host code the array's name is only a host-side
// stand-in; this address is what kernels receive.
int static_scratch(void** ptr, const char* who) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        return fail(SWIFTLLM_ERR_DEVICE_NOT_FOUND, "%s: no current HIP device", who);
    }
    if (dev < 0 || dev >= kMaxScratchDevices) {
        return fail(SWIFTLLM_ERR_NOT_SUPPORTED, "%s: device %d beyond the %d the library tracks", who,
                    dev, kMaxScratchDevices);
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch[dev] == nullptr) {
        void* p = nullptr;
        const hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (err != hipSuccess || p == nullptr) {
            return fail(SWIFTLLM_ERR_INIT, "%s: hipGetSymbolAddress(scratch) on device %d: %s", who, dev,
                        hipGetErrorString(err));
        }
        g_scratch[dev] = p;
    }
    *ptr = g_scratch[dev];
    return SWIFTLLM_OK;
}

int decode_v2_noalloc(void* out, const void* q, const void* kc, const void* vc, const int* bt,
                      const int* ctx, float scale, const Shape& sh, int partition_size,
                      int num_blocks, hipStream_t stream, const char* who) {
    int rc = validate_decode(who, out, q, kc, vc, bt, ctx, sh);
    if (rc != SWIFTLLM_OK) return rc;
    if ((rc = validate_partition(who, partition_size)) != SWIFTLLM_OK) return rc;
    const int cus = device_cus();
    const size_t need = v2_bytes(sh, effective_partition(sh, partition_size, cus), cus);
    if (need > SWIFTLLM_HIP_NOALLOC_SCRATCH_BYTES) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER,
                    "%s: these sizes need %zu bytes of split-K scratch, more than the %zu bytes of "
                    "its static scratch; use swiftllm_hip_launch_paged_attention_v2 with a workspace",
                    who, need, static_cast<size_t>(SWIFTLLM_HIP_NOALLOC_SCRATCH_BYTES));
    }
    if ((rc = require_device()) != SWIFTLLM_OK) return rc;
    if (sh.S == 0) return ok();
    void* ws = nullptr;
    if ((rc = static_scratch(&ws, who)) != SWIFTLLM_OK) return rc;
    return decode_v2(out, ws, SWIFTLLM_HIP_NOALLOC_SCRATCH_BYTES, q, kc, vc, bt, ctx, scale, sh,
                     partition_size, num_blocks, stream, who);
}

}  // namespace
}  // namespace swiftllm

using namespace swiftllm;

extern "C" {

void launch_paged_attention_v1(void* output, void* query, void* key_cache, void* value_cache,
                               int* block_tables, int* context_lens, float scale, int num_seqs,
                               int num_heads, int num_kv_heads, int head_dim, int block_size,
                               int max_num_blocks_per_seq, hipStream_t stream) {
    const Shape sh{num_seqs, num_heads, num_kv_heads, head_dim, block_size, max_num_blocks_per_seq};
    decode_v1(output, query, key_cache, value_cache, block_tables, context_lens, scale, sh, 0,
              stream, "launch_paged_attention_v1");
}

int swiftllm_hip_launch_paged_attention_v1(void* output, const void* query, const void* key_cache,
                                           const void* value_cache, const int* block_tables,
                                           const int* context_lens, float scale, int num_seqs,
                                           int num_heads, int num_kv_heads, int head_dim,
                                           int block_size, int max_num_blocks_per_seq,
                                           int num_blocks, hipStream_t stream) {
    const Shape sh{num_seqs, num_heads, num_kv_heads, head_dim, block_size, max_num_blocks_per_seq};
    return decode_v1(output, query, key_cache, value_cache, block_tables, context_lens, scale, sh,
                     num_blocks, stream, "swiftllm_hip_launch_paged_attention_v1");
}

void launch_paged_attention_v2(void* output, void* workspace, size_t workspace_bytes, void* query,
                               void* key_cache, void* value_cache, int* block_tables,
                               int* context_lens, float scale, int num_seqs, int num_heads,
                               int num_kv_heads, int head_dim, int block_size,
                               int max_num_blocks_per_seq, int partition_size, hipStream_t stream) {
    const Shape sh{num_seqs, num_heads, num_kv_heads, head_dim, block_size, max_num_blocks_per_seq};
    decode_v2(output, workspace, workspace_bytes, query, key_cache, value_cache, block_tables,
              context_lens, scale, sh, partition_size, 0, stream, "launch_paged_attention_v2");
}

int swiftllm_hip_launch_paged_attention_v2(void* output, void* workspace, size_t workspace_bytes,
                                           const void* query, const void* key_cache,
                                           const void* value_cache, const int* block_tables,
                                           const int* context_lens, float scale, int num_seqs,
                                           int num_heads, int num_kv_heads, int head_dim,
                                           int block_size, int max_num_blocks_per_seq,
                                           int partition_size, int num_blocks, hipStream_t stream) {
    const Shape sh{num_seqs, num_heads, num_kv_heads, head_dim, block_size, max_num_blocks_per_seq};
    return decode_v2(output, workspace, workspace_bytes, query, key_cache, value_cache, block_tables,
                     context_lens, scale, sh, partition_size, num_blocks, stream,
                     "swiftllm_hip_launch_paged_attention_v2");
}

int swiftllm_hip_launch_paged_attention_v2_noalloc(void* output, const void* query,
                                                   const void* key_cache, const void* value_cache,
                                                   const int* block_tables, const int* context_lens,
                                                   float scale, int num_seqs, int num_heads,
                                                   int num_kv_heads, int head_dim, int block_size,
                                                   int max_num_blocks_per_seq, int partition_size,
                                                   int num_blocks, hipStream_t stream) {
    const Shape sh{num_seqs, num_heads, num_kv_heads, head_dim, block_size, max_num_blocks_per_seq};
    return decode_v2_noalloc(output, query, key_cache, value_cache, block_tables, context_lens,
                             scale, sh, partition_size, num_blocks, stream,
                             "swiftllm_hip_launch_paged_attention_v2_noalloc");
}

size_t swiftllm_hip_paged_attention_v2_workspace_size(int num_seqs, int num_heads, int num_kv_heads,
                                                      int head_dim, int block_size,
                                                      int max_num_blocks_per_seq,
                                                      int partition_size) {
    if (num_seqs < 0 || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads != 0 ||
        head_dim <= 0 || block_size != kBlockTokens || max_num_blocks_per_seq < 0 ||
        partition_size < 0 || partition_size % kBlockTokens != 0) {
        fail(SWIFTLLM_ERR_INVALID_PARAMETER, "swiftllm_hip_paged_attention_v2_workspace_size: bad shape");
        return 0;
    }
    const Shape sh{num_seqs, num_heads, num_kv_heads, head_dim, block_size, max_num_blocks_per_seq};
    ok();
    if (partition_size == 0) {
        int n = 0;
        const int cus = (hipGetDeviceCount(&n) == hipSuccess && n > 0) ? device_cus() : kDefaultCUs;
        // the balanced workspace also covers its partitioned fallback
        return std::max(stream_need(sh, cus).total, v2_need(sh, 512, cus).total);
    }
    int n = 0;
    const int cus = (hipGetDeviceCount(&n) == hipSuccess && n > 0) ? device_cus() : kDefaultCUs;
    return v2_need(sh, partition_size, cus).total;
}

int swiftllm_hip_workspace_clear(void* workspace, size_t bytes, hipStream_t stream) {
    if (bytes == 0) return ok();
    if (workspace == nullptr || !aligned(workspace, 4) || bytes % 4 != 0) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER,
                    "swiftllm_hip_workspace_clear: null or misaligned workspace / size");
    }
    int rc = require_device();
    if (rc != SWIFTLLM_OK) return rc;
    ClearArgs a{static_cast<uint32_t*>(workspace), bytes / 4};
    const size_t blocks = (a.words + 255) / 256;
    const unsigned grid = static_cast<unsigned>(blocks < 4096 ? blocks : 4096);
    return launched(launch(clear_kernel, dim3(grid), dim3(256), 0, stream, a),
                    "swiftllm_hip_workspace_clear");
}

int swiftllm_hip_paged_attention_decode(void* output, const void* query, const void* key_cache,
                                        const void* value_cache, const int32_t* block_tables,
                                        const int32_t* context_lens,
                                        const swiftllm_paged_attention_params* p,
                                        hipStream_t stream) {
    const char* who = "swiftllm_hip_paged_attention_decode";
    if (p == nullptr) return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: null params", who);
    const size_t lim = 0x7fffffff;
    if (p->num_seqs > lim || p->num_heads > lim || p->num_kv_heads > lim || p->head_dim > lim ||
        p->block_size > lim || p->max_context_len > lim || p->block_size == 0) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: parameter out of range", who);
    }
    const size_t mb = (p->max_context_len + p->block_size - 1) / p->block_size;
    const Shape sh{static_cast<int>(p->num_seqs), static_cast<int>(p->num_heads),
                   static_cast<int>(p->num_kv_heads), static_cast<int>(p->head_dim),
                   static_cast<int>(p->block_size), static_cast<int>(mb)};
    return decode_v1(output, query, key_cache, value_cache, block_tables, context_lens, p->scale,
                     sh, 0, stream, who);
}

int swiftllm_hip_gather_kv(const void* key_cache, const void* value_cache, const int* block_tables,
                           const int* context_lens, int seq, int kv_head, int num_kv_heads,
                           int head_dim, int block_size, int max_num_blocks_per_seq,
                           int max_context_len, void* k_out, void* v_out, hipStream_t stream) {
    const char* who = "swiftllm_hip_gather_kv";
    if (seq < 0 || num_kv_heads <= 0 || kv_head < 0 || kv_head >= num_kv_heads || head_dim <= 0 ||
        max_num_blocks_per_seq < 0 || max_context_len < 0) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: bad shape", who);
    }
    if (block_size != kBlockTokens) {
        return fail(SWIFTLLM_ERR_NOT_SUPPORTED, "%s: block_size %d (supported: 16)", who, block_size);
    }
    if (max_context_len > 0 &&
        (!key_cache || !value_cache || !block_tables || !context_lens || !k_out || !v_out)) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: null pointer", who);
    }
    int rc = require_device();
    if (rc != SWIFTLLM_OK) return rc;
    if (max_context_len == 0) return ok();
    GatherArgs a{static_cast<const uint16_t*>(key_cache), static_cast<const uint16_t*>(value_cache),
                 block_tables, context_lens, static_cast<uint16_t*>(k_out),
                 static_cast<uint16_t*>(v_out), seq, kv_head, num_kv_heads, head_dim,
                 max_num_blocks_per_seq, max_context_len};
    const size_t n = static_cast<size_t>(max_context_len) * head_dim;
    const size_t blocks = (n + 255) / 256;
    const unsigned grid = static_cast<unsigned>(blocks < 65535 ? blocks : 65535);
    return launched(launch(gather_kv_kernel, dim3(grid), dim3(256), 0, stream, a), who);
}

}  // extern "C"
