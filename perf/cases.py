"""The measured calls of this package: what a serving program asks of it, from
one short sequence to a full batch of prompts, through the entry points of
swiftllm_amd.paged_attention and swiftllm_amd.moe.

torch is imported before the library, so that both use one HIP runtime: device
buffers are torch tensors handed over as raw pointers, or DeviceArrays seen
through torch. A case fixes every size, the sequence lengths included; a seed
gives the values, the block tables and the routing.
"""

from __future__ import annotations

import math
import random

import torch

from swiftllm_amd import moe
from swiftllm_amd import paged_attention as pa
from swiftllm_amd._hip import DeviceArray

BS = 16                      # tokens per cache block
DEV = "cuda"
F16, F32, F64, I32, I64 = torch.float16, torch.float32, torch.float64, torch.int32, torch.int64

# (query heads, kv heads, head_dim): a small MHA model, 8B- and 70B-like GQA
# layers, and a wide MHA layer.
HEADS = [(8, 8, 64), (32, 8, 128), (64, 8, 128), (16, 16, 128)]


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def _heads(i: int) -> dict:
    H, Hkv, D = HEADS[i]
    return {"heads": H, "kv_heads": Hkv, "head_dim": D}


def listed() -> list[dict]:
    return [
        # A handful of short chats on a small model: launch latency is the call.
        {"name": "decode_tiny", "kind": "decode", **_heads(0), "seqs": 4, "dist": "uniform",
         "lo": 1, "hi": 256, "lens_seed": 1, "partition": -1, "write": False},
        # One user, one long document: a single sequence has to fill the GPU.
        {"name": "decode_one_long", "kind": "decode", **_heads(1), "seqs": 1, "dist": "uniform",
         "lo": 7919, "hi": 7919, "lens_seed": 2, "partition": 512, "write": False},
        # The steady state of a server: 64 chats of 512 to 4096 tokens, single pass.
        {"name": "decode_batch", "kind": "decode", **_heads(1), "seqs": 64, "dist": "uniform",
         "lo": 512, "hi": 4096, "lens_seed": 3, "partition": -1, "write": False},
        # Few very long contexts on a 70B-like layer, split over 512-token partitions.
        {"name": "decode_long_split", "kind": "decode", **_heads(2), "seqs": 8, "dist": "uniform",
         "lo": 32768, "hi": 32768, "lens_seed": 4, "partition": 512, "write": False},
        # A continuous-batching step: write each sequence's new token, then attend,
        # at the partition size PagedAttention defaults to; lengths lognormal.
        {"name": "ragged_step", "kind": "decode", **_heads(1), "seqs": 256, "dist": "lognormal",
         "lo": 1, "hi": 8192, "lens_seed": 5, "partition": 512, "write": True},
        # The K/V of a batch of new prompts going into the cache (before their prefill).
        {"name": "prompt_cache_write", "kind": "write", **_heads(1), "seqs": 12, "dist": "uniform",
         "lo": 300, "hi": 2048, "lens_seed": 6},
        # Causal attention of a full batch of long prompts.
        {"name": "prefill_batch", "kind": "prefill", **_heads(1), "seqs": 8, "dist": "uniform",
         "lo": 2048, "hi": 2048, "lens_seed": 7},
        # The prompts of mixed chat traffic: mostly short, a few long, odd lengths.
        {"name": "prefill_ragged", "kind": "prefill", **_heads(1), "seqs": 24, "dist": "lognormal",
         "lo": 1, "hi": 4096, "lens_seed": 19},
        # Routing and expert-contiguous dispatch of a prefill batch, 8 experts, top-2.
        {"name": "moe_dispatch", "kind": "dispatch", "tokens": 4096, "hidden": 4096, "experts": 8,
         "top_k": 2},
        # The whole MoE layer behind the router, for a prefill batch.
        {"name": "moe_layer_batch", "kind": "moe", "tokens": 4096, "hidden": 4096, "inter": 14336,
         "experts": 8, "top_k": 2},
        # The same layer at a decode batch: it streams the experts' weights.
        {"name": "moe_layer_decode", "kind": "moe", "tokens": 64, "hidden": 4096, "inter": 14336,
         "experts": 8, "top_k": 2},
        # Copy-on-write of forked sequences: blocks copied in every layer's caches.
        {"name": "copy_blocks", "kind": "copy", "pairs": 128, "layers": 32, "kv_heads": 8,
         "head_dim": 128},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    """An integer in [lo, hi], even over its logarithm; odd as often as even."""
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng: random.Random) -> dict:
    """One more case of the same ranges, bounded by the largest listed ones."""
    kind = rng.choice(["decode", "decode", "decode", "write", "prefill", "prefill", "dispatch",
                       "moe", "moe", "copy"])
    if kind == "decode":
        h = rng.randrange(len(HEADS))
        H, Hkv, D = HEADS[h]
        seqs = _log_int(rng, 1, 256)
        # at most 1 GiB of K and V in one call
        most = min(32768, (1 << 30) // (seqs * Hkv * D * 4))
        mode = rng.choice(["v1", "v1", "split", "split", "split", "balanced"])
        write = rng.random() < 0.4
        if rng.random() < 0.4 and most >= 4096:
            dist, lo, hi = "lognormal", 1, min(8192, most)
        else:
            hi = _log_int(rng, 16, most)
            dist, lo = "uniform", max(1, hi // rng.choice([1, 2, 8, 64]))
        if mode == "v1" and seqs * Hkv < 64:
            hi = min(hi, 4096)       # a program splits longer contexts of so few sequences
            lo = min(lo, hi)
        partition = {"v1": -1, "balanced": 0, "split": rng.choice([512, 512, 1024, 4096])}[mode]
        return {"kind": kind, **_heads(h), "seqs": seqs, "dist": dist, "lo": lo, "hi": hi,
                "lens_seed": rng.randrange(1 << 20), "partition": partition, "write": write}
    if kind in ("write", "prefill"):
        h = rng.randrange(len(HEADS))
        hi = _log_int(rng, 16, 8192)
        seqs = _log_int(rng, 1, max(1, min(64, 16384 // hi)))
        dist = rng.choice(["uniform", "lognormal"])
        return {"kind": kind, **_heads(h), "seqs": seqs, "dist": dist,
                "lo": 1 if dist == "lognormal" else max(1, hi // rng.choice([1, 2, 8])),
                "hi": hi, "lens_seed": rng.randrange(1 << 20)}
    if kind == "dispatch":
        E = rng.choice([8, 8, 16, 64])
        return {"kind": kind, "tokens": _log_int(rng, 1, 4096),
                "hidden": rng.choice([1024, 2048, 2880, 4096]), "experts": E,
                "top_k": rng.choice([1, 2, 2] if E <= 16 else [2, 6, 8])}
    if kind == "moe":
        E, hidden, inter, K = rng.choice([(8, 4096, 14336, 2), (8, 4096, 14336, 2),
                                          (16, 2048, 4096, 2), (64, 2048, 1408, 6)])
        return {"kind": kind, "tokens": _log_int(rng, 1, 4096), "hidden": hidden, "inter": inter,
                "experts": E, "top_k": K}
    return {"kind": kind, "pairs": _log_int(rng, 1, 128), "layers": rng.choice([1, 16, 32]),
            "kv_heads": 8, "head_dim": rng.choice([64, 128])}


def _lens(case: dict) -> list[int]:
    """The sequence lengths of a case; part of its size, not of its data."""
    r = random.Random(case["lens_seed"])
    lo, hi = case["lo"], case["hi"]
    if case["dist"] == "lognormal":
        median = 600.0 if case["kind"] == "decode" else 300.0
        return [min(hi, max(lo, round(math.exp(r.gauss(math.log(median), 1.0)))))
                for _ in range(case["seqs"])]
    return [r.randint(lo, hi) for _ in range(case["seqs"])]


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g: torch.Generator, *shape, std: float = 1.0) -> torch.Tensor:
    return torch.empty(shape, dtype=F16, device=DEV).normal_(0.0, std, generator=g)


class _Span:
    """A DeviceArray as torch sees it; keeps the allocation alive."""

    def __init__(self, arr: DeviceArray):
        self.arr = arr
        self.__cuda_array_interface__ = {"shape": arr.shape, "typestr": arr.dtype.str,
                                         "data": (arr.ptr, False), "version": 2}


def _view(arr: DeviceArray) -> torch.Tensor:
    return torch.as_tensor(_Span(arr), device=DEV)


def _array(t: torch.Tensor) -> DeviceArray:
    """A DeviceArray with t's contents."""
    arr = DeviceArray(tuple(t.shape), str(t.dtype).replace("torch.", ""))
    _view(arr).copy_(t)
    return arr


def _attention_inputs(case: dict, seed: int) -> dict:
    """Caches with 1.25 times the blocks in use, tables over a random
    permutation of them, and the step's own tensors."""
    g = _gen(seed)
    H, Hkv, D, S = case["heads"], case["kv_heads"], case["head_dim"], case["seqs"]
    lens = _lens(case)
    need = [(n + BS - 1) // BS for n in lens]
    MB, NB = max(need), max(1, math.ceil(1.25 * sum(need)))
    perm = torch.randperm(NB, generator=g, device=DEV).to(I32)
    ctx = torch.tensor(lens, dtype=I32, device=DEV)
    nb = torch.tensor(need, dtype=I64, device=DEV)
    col = torch.arange(MB, device=DEV)
    first = torch.cumsum(nb, 0) - nb
    bt = torch.where(col < nb[:, None], perm[(first[:, None] + col).clamp_(max=NB - 1)], 0)
    bt = bt.to(I32).contiguous()
    std = 0.5 if case["kind"] == "prefill" else 1.0
    d = dict(lens=lens, S=S, H=H, Hkv=Hkv, D=D, MB=MB, NB=NB, bt=bt, ctx=ctx,
             scale=1.0 / math.sqrt(D))
    if case["kind"] == "decode":
        d["kc"] = _normal(g, NB, Hkv, D, BS, std=std)
        d["vc"] = _normal(g, NB, Hkv, D, BS, std=std)
        d["q"] = _normal(g, S, H, D, std=std)
        pos = (ctx - 1).long()
        d["slots"] = (bt.gather(1, (pos // BS)[:, None])[:, 0] * BS + pos % BS).to(I32)
        d["key"] = _normal(g, S, Hkv, D, std=std)
        d["value"] = _normal(g, S, Hkv, D, std=std)
        return d
    T = sum(lens)
    seq = torch.repeat_interleave(torch.arange(S, device=DEV), ctx.long())
    start = torch.cumsum(ctx.long(), 0) - ctx
    pos = torch.arange(T, device=DEV) - start[seq]
    d["slots"] = (bt[seq, pos // BS].long() * BS + pos % BS).to(I32)
    d["key"] = _normal(g, T, Hkv, D, std=std)
    d["value"] = _normal(g, T, Hkv, D, std=std)
    d["kc"] = torch.zeros(NB, Hkv, D, BS, dtype=F16, device=DEV)
    d["vc"] = torch.zeros(NB, Hkv, D, BS, dtype=F16, device=DEV)
    d["T"] = T
    if case["kind"] == "prefill":
        d["q"] = _normal(g, T, H, D, std=std)
        b, o = d["slots"].long() // BS, d["slots"].long() % BS
        d["kc"][b, :, :, o] = d["key"]
        d["vc"][b, :, :, o] = d["value"]
    return d


def _moe_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    T, hidden, E = case["tokens"], case["hidden"], case["experts"]
    return dict(x=_normal(g, T, hidden),
                logits=torch.empty(T, E, dtype=F32, device=DEV).normal_(generator=g))


def _moe_weights(case: dict, seed: int) -> list[DeviceArray]:
    """gate, up [E, inter, hidden] and down [E, hidden, inter], N(0, 1 / fan-in)."""
    g = _gen(seed + 0x5EED)
    E, hidden, inter = case["experts"], case["hidden"], case["inter"]
    out = []
    for n, k in ((inter, hidden), (inter, hidden), (hidden, inter)):
        w = DeviceArray((E, n, k), "float16")
        _view(w).normal_(0.0, 1.0 / math.sqrt(k), generator=g)
        out.append(w)
    return out


def _copy_inputs(case: dict, seed: int) -> dict:
    """One pool [layers, K/V, blocks, ...]; the first `pairs` blocks of a random
    permutation are copied onto the next."""
    g = _gen(seed)
    n = case["pairs"]
    NB = math.ceil(2.5 * n)
    perm = torch.randperm(NB, generator=g, device=DEV)
    return dict(NB=NB, pairs=torch.stack([perm[:n], perm[n:2 * n]], 1).contiguous(),
                pool=_normal(g, case["layers"], 2, NB, case["kv_heads"], case["head_dim"], BS))


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind in ("decode", "write", "prefill"):
        d = _attention_inputs(case, seed)
        d["case"] = case
        if kind != "write":
            d["out"] = torch.zeros_like(d["q"])
        if kind == "decode" and case["partition"] >= 0:
            d["ws"] = pa.workspace(pa.paged_attention_v2_workspace_size(
                d["S"], d["H"], d["Hkv"], d["D"], BS, d["MB"], case["partition"]))
        return d
    if kind == "copy":
        d = _copy_inputs(case, seed)
        d["case"] = case
        d["k"] = [d["pool"][i, 0].data_ptr() for i in range(case["layers"])]
        d["v"] = [d["pool"][i, 1].data_ptr() for i in range(case["layers"])]
        return d
    d = _moe_inputs(case, seed)
    T, hidden, E, K = case["tokens"], case["hidden"], case["experts"], case["top_k"]
    s = {"case": case, "x": _array(d["x"]), "logits": _array(d["logits"])}
    if kind == "dispatch":
        s["ids"] = DeviceArray((T, K), "int32")
        s["weights"] = DeviceArray((T, K), "float32")
        s["bufs"] = b = moe.DispatchBuffers.allocate(T, E, K, hidden)
        s["outputs"] = {"ids": _view(s["ids"]), "weights": _view(s["weights"]),
                        "counts": _view(b.counts), "offsets": _view(b.offsets),
                        "x_perm": _view(b.x_perm), "inverse": _view(b.inverse),
                        "sorted_token_ids": _view(b.sorted_token_ids)}
    else:
        s["mlp"] = mlp = moe.MoeMlp(E, K, *_moe_weights(case, seed))
        b = mlp.buffers(T, hidden)
        s["outputs"] = {"out": _view(b["out"])}
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s: dict):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        if case["write"]:
            pa.launch_reshape_and_cache(s["key"].data_ptr(), s["value"].data_ptr(),
                                        s["kc"].data_ptr(), s["vc"].data_ptr(),
                                        s["slots"].data_ptr(), s["S"], s["Hkv"], s["D"], BS,
                                        num_blocks=s["NB"])
        args = (s["q"].data_ptr(), s["kc"].data_ptr(), s["vc"].data_ptr(), s["bt"].data_ptr(),
                s["ctx"].data_ptr(), s["scale"], s["S"], s["H"], s["Hkv"], s["D"], BS, s["MB"])
        if case["partition"] < 0:
            pa.paged_attention_v1(s["out"].data_ptr(), *args, num_blocks=s["NB"])
        else:
            pa.paged_attention_v2(s["out"].data_ptr(), s["ws"], *args, case["partition"],
                                  num_blocks=s["NB"])
        return {"out": s["out"], "kc": s["kc"], "vc": s["vc"]} if case["write"] else s["out"]
    if kind == "write":
        pa.launch_reshape_and_cache(s["key"].data_ptr(), s["value"].data_ptr(),
                                    s["kc"].data_ptr(), s["vc"].data_ptr(), s["slots"].data_ptr(),
                                    s["T"], s["Hkv"], s["D"], BS, num_blocks=s["NB"])
        return {"kc": s["kc"], "vc": s["vc"]}
    if kind == "prefill":
        pa.launch_paged_prefill(s["out"].data_ptr(), s["q"].data_ptr(), s["kc"].data_ptr(),
                                s["vc"].data_ptr(), s["slots"].data_ptr(), s["ctx"].data_ptr(),
                                s["scale"], s["S"], s["H"], s["Hkv"], s["D"], BS, max(s["lens"]),
                                num_blocks=s["NB"])
        return s["out"]
    if kind == "copy":
        pa.copy_blocks(s["k"], s["v"], s["pairs"].data_ptr(), case["pairs"], case["kv_heads"],
                       case["head_dim"], BS)
        return s["pool"]
    if kind == "dispatch":
        moe.moe_route_dispatch(s["logits"], s["x"], case["top_k"], s["ids"], s["weights"],
                               s["bufs"])
        return s["outputs"]
    s["mlp"].forward(s["logits"], s["x"])
    return s["outputs"]


# ---------------------------------------------------------------------------
# What one pass cannot do without
# ---------------------------------------------------------------------------
def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("decode", "write", "prefill"):
        H, Hkv, D, S = case["heads"], case["kv_heads"], case["head_dim"], case["seqs"]
        lens = _lens(case)
        T = sum(lens)
        token = 2 * Hkv * D * 2                        # K and V of one token
        if kind == "decode":
            blocks = sum((n + BS - 1) // BS for n in lens)
            return {"bytes": T * token + 4 * S * H * D + 4 * blocks + 4 * S
                    + (2 * S * token + 4 * S if case["write"] else 0),
                    "flops": 4 * T * H * D}
        if kind == "write":
            return {"bytes": 2 * T * token + 4 * T, "flops": 0}
        return {"bytes": 4 * T * H * D + T * token + 4 * T + 4 * S,
                "flops": 4 * H * D * sum(n * (n + 1) // 2 for n in lens)}
    if kind == "copy":
        block = case["kv_heads"] * case["head_dim"] * BS * 2
        return {"bytes": 2 * 2 * case["layers"] * case["pairs"] * block + 16 * case["pairs"],
                "flops": 0}
    T, hidden, E, K = case["tokens"], case["hidden"], case["experts"], case["top_k"]
    if kind == "dispatch":
        return {"bytes": 4 * T * E + 2 * T * hidden + 2 * T * K * hidden + 16 * T * K + 8 * E + 4,
                "flops": 0}
    weights = 3 * min(E, T * K) * hidden * case["inter"] * 2
    return {"bytes": weights + 4 * T * E + 4 * T * hidden,
            "flops": 6 * T * K * hidden * case["inter"]}


def tolerance(case: dict):
    """Copies are exact. Attention is one fp16 rounding of sums kept in 32 bits
    (2.1e-4 off exact()); the MoE layer rounds to fp16 three times, h, y and the
    output (3.6e-4 off); routing weights are 32-bit sums. Each is about four
    times that."""
    kind = case["kind"]
    if kind in ("write", "copy"):
        return "exact"
    if kind == "dispatch":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    if kind == "moe":
        return {"rel": 1.5e-3, "max": 1e-2}
    return {"rel": 8e-4, "max": 4e-3}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _write_exact(kc, vc, key, value, slots) -> None:
    b, o = slots.long() // BS, slots.long() % BS
    kc[b, :, :, o] = key
    vc[b, :, :, o] = value


def _attend(q, k, v, scale, first):
    """q [n, H, D] at positions first .. first + n - 1 over k, v [L, Hkv, D], in
    float64; token i sees positions up to its own."""
    n, H, D = q.shape
    L, Hkv, _ = k.shape
    G = H // Hkv
    out = torch.empty(n, H, D, dtype=F64, device=DEV)
    limit = torch.arange(first, first + n, device=DEV)
    for h in range(Hkv):
        qs = q[:, h * G:(h + 1) * G].to(F64).reshape(n * G, D)
        s = qs @ k[:, h].to(F64).t().contiguous() * scale
        s = s.view(n, G, L)
        if first + 1 < L:
            s.masked_fill_((torch.arange(L, device=DEV) > limit[:, None])[:, None], -math.inf)
        p = torch.softmax(s, -1).view(n * G, L)
        out[:, h * G:(h + 1) * G] = (p @ v[:, h].to(F64).contiguous()).view(n, G, D)
    return out


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("decode", "write", "prefill"):
        d = _attention_inputs(case, seed)
        if kind == "write" or (kind == "decode" and case["write"]):
            _write_exact(d["kc"], d["vc"], d["key"], d["value"], d["slots"])
        if kind == "write":
            return {"kc": d["kc"], "vc": d["vc"]}
        out = torch.empty(d["q"].shape, dtype=F64, device=DEV)
        at = 0
        for i, n in enumerate(d["lens"]):
            blocks = d["bt"][i, :(n + BS - 1) // BS].long()
            k = d["kc"][blocks].permute(0, 3, 1, 2).reshape(-1, d["Hkv"], d["D"])[:n]
            v = d["vc"][blocks].permute(0, 3, 1, 2).reshape(-1, d["Hkv"], d["D"])[:n]
            if kind == "decode":
                out[i] = _attend(d["q"][i:i + 1], k, v, d["scale"], n - 1)[0]
                continue
            for a in range(0, n, 1024):
                b = min(n, a + 1024)
                out[at + a:at + b] = _attend(d["q"][at + a:at + b], k[:b], v[:b], d["scale"], a)
            at += n
        return {"out": out, "kc": d["kc"], "vc": d["vc"]} if case.get("write") else out
    if kind == "copy":
        d = _copy_inputs(case, seed)
        d["pool"][:, :, d["pairs"][:, 1]] = d["pool"][:, :, d["pairs"][:, 0]]
        return d["pool"]
    d = _moe_inputs(case, seed)
    x, logits, K, E = d["x"], d["logits"].to(F64), case["top_k"], case["experts"]
    top, ids = torch.topk(logits, K, dim=-1)
    weights = torch.softmax(top, -1)
    if kind == "dispatch":
        order = torch.sort(ids.reshape(-1), stable=True).indices
        return {"ids": None, "weights": weights, "counts": None, "offsets": None,
                "x_perm": x[order // K], "inverse": None, "sorted_token_ids": None}
    gate, up, down = (_view(w) for w in _moe_weights(case, seed))
    out = torch.zeros(x.shape, dtype=F64, device=DEV)
    for e in range(E):
        t, k = (ids == e).nonzero(as_tuple=True)
        if not t.numel():
            continue
        xe = x[t].to(F64)
        h = torch.nn.functional.silu(xe @ gate[e].to(F64).t()) * (xe @ up[e].to(F64).t())
        out.index_add_(0, t, weights[t, k][:, None] * (h @ down[e].to(F64).t()))
    return {"out": out}
