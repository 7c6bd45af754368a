// KV-cache write (reshape_and_cache) for gfx950.
//
// Contract (paged_attention.cu:167-199, launcher cu:271-300): for token t
// with slot = slot_mapping[t], block b = slot / BS and offset o = slot % BS,
//   key_cache[b, h, d, o]   = key[t, h, d]
//   value_cache[b, h, d, o] = value[t, h, d]
// as bit copies. The reference launches one thread per element for
// head_dim 128 / block_size 16 only (cu:286) and would write out of bounds
// for a negative slot; here any block size and head_dim are taken, negative
// slots are skipped (padding tokens), and slots past num_blocks * BS are
// skipped when the pool size is known.
//
// Row r = h * D + d of block b is the 16 tokens of (h, d) at element
// (b * Hkv * D + r) * BS; a token's element goes to column o of it. Four rows
// make a 128-byte line (BS 16).
//
// Two kernels. reshape_and_cache_runs_kernel takes block size 16: it finds
// the runs of consecutive slots (a prompt fills whole blocks), transposes
// them through LDS and writes whole rows, so a block's lines are written
// once. reshape_and_cache_kernel takes every other block size, row count and
// alignment, one workgroup per token. Both write a lone token's column with
// consecutive lanes on consecutive rows: one wave store instruction covers 16
// whole lines with 8 bytes each, where a lane per 4 consecutive d (four
// stores to the 4 rows of one line) needs 64 lines per instruction and four
// instructions per line. Measured alone on MI355X (the stores of 256 tokens
// of 8 kv heads x 128, no loads): 8.7 us against 23.4 us.

#include "common.hpp"

namespace swiftllm {
namespace {

struct CacheArgs {
    const uint16_t* key;
    const uint16_t* value;
    uint16_t* kc;
    uint16_t* vc;
    const int* slots;
    long long key_stride;    // elements between consecutive tokens of key
    long long value_stride;  // elements between consecutive tokens of value
    long long num_slots;     // num_blocks * BS, or <= 0 when unknown
    int T;
    int Hkv;
    int D;
    int BS;
};

// Each store is 2 bytes of a 32-byte tile row, so the memory system merges
// it into the row (a read-modify-write below the caches). Nontemporal stores
// do that inside this kernel. Cached stores leave partly dirty lines that are
// written back while the next kernel (the decode) streams the pool, and
// writes mixed into that read stream cost it more than this kernel's own
// time (config 4: 21 us here and no decode slowdown, against 9 us here and
// 10-17 us added to the decode).
__device__ __forceinline__ void put(uint16_t* p, uint16_t v) {
    __builtin_nontemporal_store(v, p);
}

// Rows per thread per pass: a pass of 256 threads covers 1024 rows, all of
// Llama-3-8B's Hkv * D; its 8 loads per thread are issued before any store.
constexpr int kRowsPerThread = 4;

__global__ __launch_bounds__(256) void reshape_and_cache_kernel(const CacheArgs a) {
    const int t = blockIdx.x;
    const int slot = a.slots[t];
    if (slot < 0 || (a.num_slots > 0 && slot >= a.num_slots)) return;
    const int b = slot / a.BS;
    const int o = slot - b * a.BS;
    const int n = a.Hkv * a.D;
    const uint16_t* kr = a.key + t * a.key_stride;
    const uint16_t* vr = a.value + t * a.value_stride;
    uint16_t* kdst = a.kc + static_cast<size_t>(b) * n * a.BS + o;
    uint16_t* vdst = a.vc + static_cast<size_t>(b) * n * a.BS + o;
    for (int r0 = 0; r0 < n; r0 += 256 * kRowsPerThread) {
        uint16_t kv[kRowsPerThread], vv[kRowsPerThread];
#pragma unroll
        for (int i = 0; i < kRowsPerThread; ++i) {
            const int r = r0 + i * 256 + threadIdx.x;
            if (r < n) {
                kv[i] = kr[r];
                vv[i] = vr[r];
            }
        }
#pragma unroll
        for (int i = 0; i < kRowsPerThread; ++i) {
            const int r = r0 + i * 256 + threadIdx.x;
            if (r < n) {
                put(kdst + static_cast<size_t>(r) * a.BS, kv[i]);
                put(vdst + static_cast<size_t>(r) * a.BS, vv[i]);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Runs of tokens (block size 16).
//
// Bound: HBM, one read of the new K/V and one write of the blocks. Column
// stores write a row's 32 bytes in 16 partial writes, each a
// read-modify-write below the caches: 16384 prompt tokens of 8 x 128 took
// 506 us (0.27 TB/s) token by token and take 21.8 us (6.2 TB/s) in runs; 600
// tokens 21.2 -> 3.9 us.
//
// A workgroup owns the runs whose first token lies in its window of W tokens,
// for 256 rows of K or of V: 16 x 512 bytes in, 8 KiB of whole lines out. The
// small piece keeps a short call parallel (a 256-token decode step is 512
// workgroups) and a long one at several workgroups per CU. Runs are cut at
// block ends only, never at a window's, so a full block is always one piece,
// wherever a prompt starts in the batch.
// ---------------------------------------------------------------------------
typedef short s4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s4v lds_s4v;
typedef unsigned u4v __attribute__((ext_vector_type(4)));

constexpr int kWinRows = 256;                  // rows (h, d) of K or V per workgroup
constexpr int kWinStride = kWinRows + 16;      // halves per token in LDS (544 bytes)

// W: tokens whose runs a workgroup owns, at most 16 (one lane of 32 looks at
// each of the W + 15 tokens those runs can span).
template <int W>
__global__ __launch_bounds__(256) void reshape_and_cache_runs_kernel(const CacheArgs a) {
    constexpr int kMax = W + kBlockTokens - 1;
    constexpr int kLoads = (kMax + 7) / 8;     // 16-byte loads per lane, 8 tokens each
    __shared__ __align__(16) uint16_t tile[kMax * kWinStride];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = a.Hkv * a.D;
    const int row0 = blockIdx.y * kWinRows;
    const int t0 = blockIdx.x * W;
    const bool is_v = blockIdx.z != 0;

    // Lane i classifies token t0 + i: a valid token continues the run of the
    // token before it when its slot is the next one of the same block, else
    // it is a run's head.
    const int t = t0 + lane;
    int slot = -1, prev = -1;
    if (lane <= kMax && t < a.T) {
        slot = a.slots[t];
        if (t > 0) prev = a.slots[t - 1];
    }
    const bool valid = slot >= 0 && (a.num_slots <= 0 || slot < a.num_slots);
    const bool cont = valid && (slot & (kBlockTokens - 1)) != 0 && prev == slot - 1;
    const unsigned conts = static_cast<unsigned>(__ballot(cont));
    unsigned heads = static_cast<unsigned>(__ballot(valid && !cont)) & ((1u << W) - 1u);
    if (heads == 0) return;  // the same in every wave
    uint16_t* const cache = is_v ? a.vc : a.kc;
    const uint16_t* const src = (is_v ? a.value : a.key) + row0;
    const long long stride = is_v ? a.value_stride : a.key_stride;
    if ((conts & (heads << 1)) == 0) {
        // Every head is a lone token (a decode step): one column each, lanes
        // on consecutive rows as in the token kernel, all loads first.
        if (row0 + tid >= n) return;
        uint16_t v[W];
#pragma unroll
        for (int i = 0; i < W; ++i) v[i] = src[min(t0 + i, a.T - 1) * stride + tid];
#pragma unroll
        for (int i = 0; i < W; ++i) {
            if ((heads >> i) & 1u) {
                const int s = __builtin_amdgcn_readlane(slot, i);
                put(cache + (static_cast<size_t>(s >> kBlockShift) * n + row0 + tid) * kBlockTokens +
                        (s & (kBlockTokens - 1)),
                    v[i]);
            }
        }
        return;
    }
    const int first = __builtin_ctz(heads);
    const int last = 31 - __builtin_clz(heads);
    // A run never passes its block's end, so it has at most 16 tokens and
    // lane last + 16 <= W + 15 does not continue it.
    const int end = last + 1 + __builtin_ctz(~(conts >> (last + 1)));

    // Tokens first .. end - 1 of the window into LDS, [token][row].
    const int c = (tid & 31) * 8;
    u4v buf[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int k = first + 8 * i + (tid >> 5);
        if (k < end && row0 + c < n) {
            buf[i] = *reinterpret_cast<const u4v*>(src + (t0 + k) * stride + c);
        }
    }
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int k = 8 * i + (tid >> 5);
        if (first + k < end) *reinterpret_cast<u4v*>(tile + k * kWinStride + c) = buf[i];
    }
    __syncthreads();

    const int r = lane & 15;
    const int kg = lane >> 4;
    for (; heads != 0; heads &= heads - 1) {
        const int i = __builtin_ctz(heads);
        const int len = 1 + __builtin_ctz(~(conts >> (i + 1)));
        const int s = __builtin_amdgcn_readlane(slot, i);
        const int o = s & (kBlockTokens - 1);
        uint16_t* const dst = cache + (static_cast<size_t>(s >> kBlockShift) * n + row0) * kBlockTokens;
        const uint16_t* const from = tile + (i - first) * kWinStride;
        if (len == 1) {
            // One column: lanes on consecutive rows (see the token kernel).
            if (row0 + tid < n) put(dst + tid * kBlockTokens + o, from[tid]);
            continue;
        }
        // Lane (r, kg) takes tokens 4 kg .. 4 kg + 3 of row r of each group
        // of 16 rows: ds_read_b64_tr_b16 hands lane i of 16 the element i % 4
        // of lanes i / 4, + 4, + 8 and + 12, so those lanes read 4 rows each
        // of 4 tokens. Columns outside the run read some staged token.
        const int col = 4 * kg + (r >> 2) - o;
        const uint16_t* const mine =
            from + min(max(col, 0), len - 1) * kWinStride + 4 * (r & 3);
        const int lo = max(o - 4 * kg, 0), hi = min(o + len - 4 * kg, 4);
#pragma unroll
        for (int g = 0; g < kWinRows / 64; ++g) {
            const int rg = 16 * (4 * g + w);
            if (row0 + rg >= n) break;
            const s4v v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds_s4v*)(const_cast<uint16_t*>(mine) + rg));
            uint16_t* const p = dst + (rg + r) * kBlockTokens + 4 * kg;
            if (lo <= 0 && hi >= 4) {
                __builtin_nontemporal_store(v, reinterpret_cast<s4v*>(p));
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (j >= lo && j < hi) put(p + j, static_cast<uint16_t>(v[j]));
                }
            }
        }
    }
}

// Up to here a call is a decode step or a few short prompts, and windows of 4
// tokens keep enough workgroups: 64 lone tokens of 8 x 128 take 4.5-5.1 us in
// windows of 4 and 6.4 us in windows of 16 (5.3 us token by token), 256 take
// 9.2 and 10.0 (9.5). Past it windows of 16 leave fewer workgroups that find
// no head: 1024 lone tokens take 29.0 us with them (29.6 token by token).
// A layer of few rows leaves few workgroups at any window, and short runs pay
// for it, one after the other in a window: up to kSmallPieces tokens times
// slices of 256 rows it keeps windows of 4. Measured in runs of 2 tokens,
// windows of 4 / 16 (token by token): 513 tokens of 2 x 128 5.4 / 9.8 (6.2),
// of 1 x 128 4.0 / 6.8 (4.7), 1024 of 2 x 128 6.8 / 9.9 (9.1), 2048 12.5 / 12.2
// (15.6); in one run 1024 of 2 x 128 3.8 / 4.0, of 8 x 64 4.4 / 3.9.
constexpr int kSmallTokens = 512;
constexpr long long kSmallPieces = 1024;

int reshape_and_cache(const void* key, const void* value, void* key_cache, void* value_cache,
                      const int* slot_mapping, int num_tokens, int num_kv_heads, int head_dim,
                      int block_size, int num_blocks, hipStream_t stream, const char* who) {
    if (num_tokens < 0 || num_kv_heads <= 0 || head_dim <= 0 || block_size <= 0) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER,
                    "%s: num_tokens=%d num_kv_heads=%d head_dim=%d block_size=%d", who, num_tokens,
                    num_kv_heads, head_dim, block_size);
    }
    if (num_tokens > 0 && (!key || !value || !key_cache || !value_cache || !slot_mapping)) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: null pointer", who);
    }
    if (!aligned(key, 2) || !aligned(value, 2) || !aligned(key_cache, 2) ||
        !aligned(value_cache, 2) || !aligned(slot_mapping, 4)) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: misaligned pointer", who);
    }
    int rc = require_device();
    if (rc != SWIFTLLM_OK) return rc;
    if (num_tokens == 0) return ok();
    CacheArgs a{};
    a.key = static_cast<const uint16_t*>(key);
    a.value = static_cast<const uint16_t*>(value);
    a.kc = static_cast<uint16_t*>(key_cache);
    a.vc = static_cast<uint16_t*>(value_cache);
    a.slots = slot_mapping;
    a.key_stride = static_cast<long long>(num_kv_heads) * head_dim;  // cu:294
    a.value_stride = a.key_stride;                                   // cu:295
    a.num_slots = num_blocks > 0 ? static_cast<long long>(num_blocks) * block_size : 0;
    a.T = num_tokens;
    a.Hkv = num_kv_heads;
    a.D = head_dim;
    a.BS = block_size;
    const long long n = static_cast<long long>(num_kv_heads) * head_dim;
    const long long slices = (n + kWinRows - 1) / kWinRows;
    const int W = num_tokens <= kSmallTokens || num_tokens * slices <= kSmallPieces ? 4 : 16;
    const long long windows = (static_cast<long long>(num_tokens) + W - 1) / W;
    if (block_size == kBlockTokens && n % 16 == 0 && windows < (1 << 24) && slices <= 65535 &&
        aligned(key, 16) && aligned(value, 16) && aligned(key_cache, 8) && aligned(value_cache, 8)) {
        const dim3 grid(static_cast<unsigned>(windows), static_cast<unsigned>(slices), 2);
        return launched(launch(W == 4 ? reshape_and_cache_runs_kernel<4>
                                      : reshape_and_cache_runs_kernel<16>,
                               grid, dim3(256), 0, stream, a),
                        who);
    }
    return launched(launch(reshape_and_cache_kernel, dim3(num_tokens), dim3(256), 0, stream, a),
                    who);
}

}  // namespace
}  // namespace swiftllm

using namespace swiftllm;

extern "C" {

void launch_reshape_and_cache(void* key, void* value, void* key_cache, void* value_cache,
                              int* slot_mapping, int num_tokens, int num_kv_heads, int head_dim,
                              int block_size, hipStream_t stream) {
    reshape_and_cache(key, value, key_cache, value_cache, slot_mapping, num_tokens, num_kv_heads,
                      head_dim, block_size, 0, stream, "launch_reshape_and_cache");
}

int swiftllm_hip_launch_reshape_and_cache(const void* key, const void* value, void* key_cache,
                                          void* value_cache, const int* slot_mapping,
                                          int num_tokens, int num_kv_heads, int head_dim,
                                          int block_size, int num_blocks, hipStream_t stream) {
    return reshape_and_cache(key, value, key_cache, value_cache, slot_mapping, num_tokens,
                             num_kv_heads, head_dim, block_size, num_blocks, stream,
                             "swiftllm_hip_launch_reshape_and_cache");
}

int swiftllm_hip_reshape_and_cache(const void* key, const void* value, void* key_cache,
                                   void* value_cache, const int32_t* slot_mapping,
                                   const swiftllm_reshape_cache_params* p, hipStream_t stream) {
    const char* who = "swiftllm_hip_reshape_and_cache";
    if (p == nullptr) return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: null params", who);
    const size_t lim = 0x7fffffff;
    if (p->num_tokens > lim || p->num_kv_heads > lim || p->head_dim > lim || p->block_size > lim) {
        return fail(SWIFTLLM_ERR_INVALID_PARAMETER, "%s: parameter out of range", who);
    }
    return reshape_and_cache(key, value, key_cache, value_cache, slot_mapping,
                             static_cast<int>(p->num_tokens), static_cast<int>(p->num_kv_heads),
                             static_cast<int>(p->head_dim), static_cast<int>(p->block_size), 0,
                             stream, who);
}

}  // extern "C"
