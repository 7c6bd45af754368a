"""Paged prefill on the GPU against oracle.prefill_numpy (float64), to the
attention tolerance (max_abs <= 2e-3, max_rel <= 1e-2 with a 1e-3 floor):
packed prompts of ragged lengths around block edges, GQA groups from 1 to
32, head_dim 64 and 128, NaN in every unused cache slot, the bounded status
entry, the bindings twin and PagedAttention.prefill."""

import dataclasses

import numpy as np
import pytest

import oracle
from helpers import assert_attention_close
from swiftllm_amd import paged_attention as pa
from swiftllm_amd import workloads
from swiftllm_amd._hip import DeviceArray, synchronize

pytestmark = pytest.mark.gpu


def _run(w, entry="status", max_len=None):
    T, H, D = w.q.shape
    Hkv = w.key_cache.shape[1]
    S = len(w.context_lens)
    max_len = int(w.context_lens.max()) if max_len is None else max_len
    out = DeviceArray((T, H, D), np.float16)
    out.fill_byte(0xFF)
    q = DeviceArray.from_numpy(w.q)
    kc, vc = DeviceArray.from_numpy(w.key_cache), DeviceArray.from_numpy(w.value_cache)
    sm, ctx = DeviceArray.from_numpy(w.slot_mapping), DeviceArray.from_numpy(w.context_lens)
    if entry == "status":
        pa.launch_paged_prefill(out, q, kc, vc, sm, ctx, w.scale, S, H, Hkv, D, 16, max_len,
                                num_blocks=w.key_cache.shape[0])
    else:
        pa.paged_attention_prefill(out, q, kc, vc, sm, ctx,
                                   pa.PagedAttentionParams(S, H, Hkv, D, 16, w.scale, max_len))
    synchronize()
    return out.numpy()


def _ref(w):
    return oracle.prefill_numpy(w.q, w.key_cache, w.value_cache, w.slot_mapping, w.context_lens,
                                w.scale)


@pytest.mark.parametrize("H,Hkv,D", [(32, 8, 128), (8, 8, 64), (64, 8, 128), (16, 1, 64),
                                     (32, 1, 128), (12, 4, 64)])
def test_prefill_gqa_shapes(dev, H, Hkv, D):
    lens = (1, 15, 16, 17, 70, 129)
    w = workloads.prefill_config(lens, H, Hkv, D, seed=H * 10 + Hkv + D)
    assert_attention_close(_run(w), _ref(w), f"prefill H{H} Hkv{Hkv} D{D}")


@pytest.mark.parametrize("entry", ["status", "params"])
def test_prefill_long_prompts(dev, entry):
    """Llama-3-8B layer heads, two long prompts and a short one."""
    w = workloads.prefill_config((1024, 517, 3), 32, 8, 128, seed=7)
    assert_attention_close(_run(w, entry), _ref(w), f"prefill long {entry}")


@pytest.mark.parametrize("H,Hkv,D", [(32, 8, 128), (16, 4, 64)])
def test_prefill_walks_past_two_id_chunks(dev, H, Hkv, D):
    """Key walks of more than 128 blocks: the kernel keeps the block ids of
    its walk in chunks of 64 blocks, double-buffered, so a 2600-token prompt
    crosses into the second chunk and reuses the first chunk's buffer for the
    third; 1100 tokens end just past the first chunk; 5 is a one-block walk."""
    w = workloads.prefill_config((2600, 1100, 5), H, Hkv, D, seed=21 + D)
    assert_attention_close(_run(w), _ref(w), f"prefill id chunks H{H} Hkv{Hkv} D{D}")


@pytest.mark.parametrize("scale", [-0.0883883, 0.0, 0.3])
def test_prefill_scale_signs(dev, scale):
    """A positive scale takes the kernel's path with the scale folded into the
    exp2 argument (max on unscaled scores); zero and negative scales take the
    plain path (max on scaled scores). Both against the oracle."""
    w = dataclasses.replace(workloads.prefill_config((1, 17, 70, 129), 32, 8, 128, seed=11),
                            scale=scale)
    assert_attention_close(_run(w), _ref(w), f"prefill scale {scale}")


def test_prefill_key_cache_8_byte_aligned(dev):
    """A key cache that is 8- but not 16-byte aligned takes the kernel's
    register path for K (the default path copies K tiles into LDS with
    16-byte loads); both against the oracle."""
    w = workloads.prefill_config((1, 17, 70, 129), 32, 8, 128, seed=13)
    T, H, D = w.q.shape
    S = len(w.context_lens)
    kc_buf = DeviceArray((w.key_cache.nbytes + 16,), np.uint8)
    kc_bytes = np.zeros(w.key_cache.nbytes + 16, np.uint8)
    kc_bytes[8:8 + w.key_cache.nbytes] = w.key_cache.view(np.uint8).ravel()
    kc_buf.upload(kc_bytes)
    out = DeviceArray((T, H, D), np.float16)
    q = DeviceArray.from_numpy(w.q)
    vc = DeviceArray.from_numpy(w.value_cache)
    sm, ctx = DeviceArray.from_numpy(w.slot_mapping), DeviceArray.from_numpy(w.context_lens)
    pa.launch_paged_prefill(out, q, kc_buf.ptr + 8, vc, sm, ctx, w.scale, S, H, 8, D, 16,
                            int(w.context_lens.max()), num_blocks=w.key_cache.shape[0])
    synchronize()
    assert_attention_close(out.numpy(), _ref(w), "prefill, key cache at +8 bytes")


def test_prefill_empty_and_zero_length_sequences(dev):
    w = workloads.prefill_config((0, 33, 0, 5), 8, 2, 64, seed=8)
    out = _run(w)
    assert_attention_close(out, _ref(w), "prefill with empty prompts")


def test_prefill_grid_rounds_past_65535(dev):
    """65535 one-token prompts with 16 kv heads: 1,048,560 (sequence, kv head)
    units, so the launch needs 131,070 rounds of 8 units, more than one grid
    row (65535) holds, and the second grid plane runs. A one-token prompt
    attends only to itself: out = its own V (the prompts share a pool of 64
    blocks; slots 1..15 of every block hold NaN)."""
    S, H, Hkv, D, NB = 65535, 16, 16, 64, 64
    rng = np.random.default_rng(5)
    q = (rng.standard_normal((S, H, D)) * 0.5).astype(np.float16)
    kc = np.full((NB, Hkv, D, 16), np.nan, np.float16)
    vc = np.full((NB, Hkv, D, 16), np.nan, np.float16)
    kc[:, :, :, 0] = (rng.standard_normal((NB, Hkv, D)) * 0.5).astype(np.float16)
    vc[:, :, :, 0] = (rng.standard_normal((NB, Hkv, D)) * 0.5).astype(np.float16)
    block = np.arange(S, dtype=np.int32) % NB
    slots = (block * 16).astype(np.int32)
    ctx = np.ones(S, np.int32)
    out = DeviceArray((S, H, D), np.float16)
    out.fill_byte(0xFF)
    pa.launch_paged_prefill(out, DeviceArray.from_numpy(q), DeviceArray.from_numpy(kc),
                            DeviceArray.from_numpy(vc), DeviceArray.from_numpy(slots),
                            DeviceArray.from_numpy(ctx), 1.0 / 8.0, S, H, Hkv, D, 16, 1,
                            num_blocks=NB)
    synchronize()
    expect = vc[block, :, :, 0]  # [S, Hkv, D]; G = 1: head h reads kv head h
    assert_attention_close(out.numpy(), expect, "prefill 65535 one-token prompts")


def test_prefill_max_len_above_every_prompt(dev):
    """A generous max_context_len only adds workgroups that exit at once."""
    w = workloads.prefill_config((20, 50), 8, 2, 64, seed=9)
    assert_attention_close(_run(w, max_len=4096), _ref(w), "prefill max_len 4096")


def test_prefill_out_of_pool_blocks_are_skipped(dev):
    """With the pool bound, a prompt whose slots point past the pool reads
    nothing out of bounds; its outputs stay finite and the others are exact."""
    w = workloads.prefill_config((40, 24), 8, 2, 64, seed=10)
    NB = w.key_cache.shape[0]
    w.slot_mapping[40:] = (NB + 3) * 16 + np.arange(24) % 16   # second prompt: outside the pool
    out = _run(w)
    ref = _ref_first(w, 40)
    assert_attention_close(out[:40], ref, "prefill in-pool prompt")
    assert np.all(np.isfinite(out[40:].astype(np.float64)))


@pytest.mark.parametrize("key_offset", [0, 8])
def test_prefill_padding_slots_attend_nothing(dev, key_offset):
    """A prompt whose slots are -1 (padding, as reshape_and_cache skips them)
    reads no block: -1 // 16 must not become block 0. Its rows attend to no
    key and come out as zeros; the prompts beside it are exact. key_offset 8
    runs the register path for K, 0 the LDS path."""
    w = workloads.prefill_config((40, 24, 19), 8, 2, 64, seed=12)
    w.slot_mapping[40:64] = -1
    T, H, D = w.q.shape
    S = len(w.context_lens)
    kc_buf = DeviceArray((w.key_cache.nbytes + 16,), np.uint8)
    kc_bytes = np.zeros(w.key_cache.nbytes + 16, np.uint8)
    kc_bytes[key_offset:key_offset + w.key_cache.nbytes] = w.key_cache.view(np.uint8).ravel()
    kc_buf.upload(kc_bytes)
    out = DeviceArray((T, H, D), np.float16)
    out.fill_byte(0xFF)
    sm, ctx = DeviceArray.from_numpy(w.slot_mapping), DeviceArray.from_numpy(w.context_lens)
    pa.launch_paged_prefill(out, DeviceArray.from_numpy(w.q), kc_buf.ptr + key_offset,
                            DeviceArray.from_numpy(w.value_cache), sm, ctx, w.scale, S, H, 2, D, 16,
                            int(w.context_lens.max()), num_blocks=w.key_cache.shape[0])
    synchronize()
    got = out.numpy()
    assert np.array_equal(got[40:64].view(np.uint16), np.zeros((24, H, D), np.uint16))
    ref_a = oracle.prefill_numpy(w.q[:40], w.key_cache, w.value_cache, w.slot_mapping[:40],
                                 w.context_lens[:1], w.scale)
    ref_c = oracle.prefill_numpy(w.q[64:], w.key_cache, w.value_cache, w.slot_mapping[64:],
                                 w.context_lens[2:], w.scale)
    assert_attention_close(got[:40], ref_a, "prefill prompt before the padding")
    assert_attention_close(got[64:], ref_c, "prefill prompt after the padding")


def _ref_first(w, n):
    return oracle.prefill_numpy(w.q[:n], w.key_cache, w.value_cache, w.slot_mapping[:n],
                                w.context_lens[:1], w.scale)


def test_paged_attention_prefill_op(dev):
    """PagedAttention.prefill (paged_attention.rs:154-189): stores K/V through
    slot_mapping, then the causal attention; query [B, S, H, D]."""
    B, S, H, Hkv, D = 3, 37, 8, 2, 64
    w = workloads.prefill_config((S,) * B, H, Hkv, D, seed=11, poison=True)
    kc0 = np.full_like(w.key_cache, np.nan)
    vc0 = np.full_like(w.value_cache, np.nan)
    op = pa.PagedAttention(pa.PagedAttentionConfig.new(H, Hkv, D, 16))
    kc, vc = DeviceArray.from_numpy(kc0), DeviceArray.from_numpy(vc0)
    out = op.prefill(DeviceArray.from_numpy(w.q.reshape(B, S, H, D)),
                     DeviceArray.from_numpy(w.key.reshape(B, S, Hkv, D)),
                     DeviceArray.from_numpy(w.value.reshape(B, S, Hkv, D)),
                     kc, vc, list(w.slot_mapping))
    assert out.shape == (B, S, H, D)
    assert_attention_close(out.numpy().reshape(B * S, H, D), _ref(w), "PagedAttention.prefill")
    b, o = w.slot_mapping // 16, w.slot_mapping % 16
    assert np.array_equal(kc.numpy()[b, :, :, o].view(np.uint16), w.key.view(np.uint16))


@pytest.mark.parametrize("H,Hkv,D", [(8, 8, 128), (6, 2, 64), (10, 2, 128), (24, 1, 128), (40, 1, 64),
                                     (66, 2, 128), (32, 16, 64)])
def test_prefill_tiles_around_stage_ends(dev, H, Hkv, D):
    """Rows per wave of 32 tokens x 1 head to 1 token x 32 heads (and chunks of
    32 heads whose second is 8 or 1 wide), kv heads that do and do not divide
    over the 8 XCDs, prompts that end on, before and after a 64-key stage, and
    walks past one and two chunks of 64 block ids."""
    lens = (63, 64, 65, 0, 127, 128, 129, 1023, 1024, 1041, 1, 2100)
    if H * D > 4096:
        lens = (63, 64, 65, 0, 129, 1, 1041)
    w = workloads.prefill_config(lens, H, Hkv, D, seed=H + Hkv + D)
    assert_attention_close(_run(w, max_len=5000), _ref(w), f"prefill tiles H{H} Hkv{Hkv} D{D}")


@pytest.mark.parametrize("S,top", [(64, 300), (65, 300), (1024, 40), (1025, 40)])
def test_prefill_tile_list(dev, S, top):
    """Sequence counts around the register and LDS tables of the work list and
    its limit, with more tiles than the grid holds workgroups and many prompts
    of equal length."""
    rng = np.random.default_rng(S)
    lens = rng.integers(0, top, size=S)
    lens[rng.choice(S, size=S // 4, replace=False)] = top
    w = workloads.prefill_config(lens, 8, 8, 64, seed=S)
    assert_attention_close(_run(w), _ref(w), f"prefill S={S}")


@pytest.mark.parametrize("shift", ["q", "out", "value_cache"])
def test_prefill_8_byte_aligned_arrays(dev, shift):
    """q, out or the value cache 8 bytes past a 16-byte boundary."""
    w = workloads.prefill_config((1, 17, 70, 129), 32, 8, 128, seed=17)
    T, H, D = w.q.shape
    arrays = {"q": w.q, "out": np.full_like(w.q, np.nan), "key_cache": w.key_cache,
              "value_cache": w.value_cache}
    bufs = {k: DeviceArray((a.size + 8,), np.float16) for k, a in arrays.items()}
    at = {k: 8 if k == shift else 0 for k in arrays}
    for k, a in arrays.items():
        bufs[k].upload_at(at[k], a)
    p = {k: bufs[k].ptr + at[k] for k in arrays}
    sm, ctx = DeviceArray.from_numpy(w.slot_mapping), DeviceArray.from_numpy(w.context_lens)
    pa.launch_paged_prefill(p["out"], p["q"], p["key_cache"], p["value_cache"], sm, ctx, w.scale,
                            len(w.context_lens), H, 8, D, 16, int(w.context_lens.max()),
                            num_blocks=w.key_cache.shape[0])
    synchronize()
    out = bufs["out"].download_at(at["out"], w.q.shape, np.float16)
    assert_attention_close(out, _ref(w), f"prefill, {shift} at +8 bytes")


@pytest.mark.parametrize("H,Hkv,D", [(8, 8, 64), (8, 8, 128), (8, 4, 128)])
def test_prefill_first_block_out_of_pool(dev, H, Hkv, D):
    """The first block of a prompt outside the pool: the rows of a wave's 32
    that see only that block attend to no key and come out as zeros, beside
    rows of the same wave that see the next block. The others attend to the
    keys from position 16 on, as a prompt that starts there would."""
    L = 120
    w = workloads.prefill_config((L, 33), H, Hkv, D, seed=31 + D)
    w.slot_mapping[:16] = -1
    out = _run(w)
    assert np.array_equal(out[:16].view(np.uint16), np.zeros((16, H, D), np.uint16))
    ref = oracle.prefill_numpy(w.q[16:], w.key_cache, w.value_cache, w.slot_mapping[16:],
                               np.array([L - 16, 33]), w.scale)
    assert_attention_close(out[16:], ref, f"prefill first block out H{H} Hkv{Hkv} D{D}")


@pytest.mark.parametrize("H,Hkv,D,lens", [
    (8, 8, 64, (96, 5)), (8, 8, 64, (97, 5)),             # rows at and past the line, few tiles
    (32, 8, 128, (24, 0, 1)), (32, 8, 128, (25, 0, 1)),
    (40, 1, 128, (2, 1)), (40, 1, 128, (3, 1)),
    (16, 16, 128, (32, 1) * 20), (16, 16, 128, (33, 1) * 20),   # more tiles than the grid holds
])
def test_prefill_prompts_of_a_few_tokens(dev, H, Hkv, D, lens):
    """The line between the per-wave and the shared-stage kernel."""
    w = workloads.prefill_config(lens, H, Hkv, D, seed=H + max(lens))
    assert_attention_close(_run(w), _ref(w), f"prefill H{H} Hkv{Hkv} D{D} up to {max(lens)}")


def _run_key_offset(w, key_offset):
    """_run with the key cache key_offset bytes past a 16-byte boundary."""
    T, H, D = w.q.shape
    kc = DeviceArray((w.key_cache.size + 8,), np.float16)
    kc.upload_at(key_offset, w.key_cache)
    out = DeviceArray((T, H, D), np.float16)
    out.fill_byte(0xFF)
    q, vc = DeviceArray.from_numpy(w.q), DeviceArray.from_numpy(w.value_cache)
    sm, ctx = DeviceArray.from_numpy(w.slot_mapping), DeviceArray.from_numpy(w.context_lens)
    pa.launch_paged_prefill(out, q, kc.ptr + key_offset, vc, sm, ctx, w.scale, len(w.context_lens), H,
                            w.key_cache.shape[1], D, 16, int(w.context_lens.max()),
                            num_blocks=w.key_cache.shape[0])
    synchronize()
    return out.numpy()


@pytest.mark.parametrize("H,Hkv,D,L,sign,key_offset", [
    (6, 2, 64, 30, 1, 0), (6, 2, 128, 30, 1, 0), (10, 2, 128, 19, 1, 0),  # prompts of a few tokens
    (6, 2, 64, 120, -1, 0), (10, 2, 128, 120, -1, 0),                     # a negative scale
    (6, 2, 128, 120, 1, 8), (10, 2, 64, 120, 1, 8), (10, 2, 64, 120, -1, 8),  # K through registers
])
def test_prefill_first_block_out_of_pool_per_wave(dev, H, Hkv, D, L, sign, key_offset):
    """The same in the per-wave kernel, on each of its calls: with 3 or 5 heads
    to a kv head a group of 16 query rows holds tokens of the first block
    (which see no key) and of the second, whose maxima rescale the group."""
    w = workloads.prefill_config((L, 13), H, Hkv, D, seed=37 + D + L)
    w = dataclasses.replace(w, scale=sign * w.scale)
    w.slot_mapping[:16] = -1
    out = _run_key_offset(w, key_offset)
    assert np.array_equal(out[:16].view(np.uint16), np.zeros((16, H, D), np.uint16))
    ref = oracle.prefill_numpy(w.q[16:], w.key_cache, w.value_cache, w.slot_mapping[16:],
                               np.array([L - 16, 13]), w.scale)
    assert_attention_close(out[16:], ref, f"prefill first block out H{H} Hkv{Hkv} D{D} L{L}")


@pytest.mark.parametrize("H,Hkv,D", [(8, 8, 64), (8, 8, 128), (8, 4, 64), (6, 2, 128), (32, 8, 128),
                                     (64, 8, 64)])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_prefill_non_finite_value_stays_near_its_token(dev, H, Hkv, D, bad):
    """A value that is not finite reaches the tokens that attend to it and, as
    0 times it is NaN, earlier ones of the same wave: at most 32 tokens that
    end in its block or later. Tokens before 80 share no wave with one past 95
    (32 or 16 tokens a wave, aligned, or at most 10), so token 100 of a
    300-token prompt leaves them as they are, whatever a workgroup spans."""
    w = workloads.prefill_config((300,), H, Hkv, D, seed=41 + D)
    ref = _ref(w)
    b, o = w.slot_mapping[100] // 16, w.slot_mapping[100] % 16
    w.value_cache[b, :, :, o] = bad
    for sign in (1, -1):
        v = dataclasses.replace(w, scale=sign * w.scale)
        if sign < 0:
            ref = oracle.prefill_numpy(w.q[:96], w.key_cache, w.value_cache, w.slot_mapping[:96],
                                       np.array([96]), v.scale)
        out = _run(v)
        assert_attention_close(out[:80], ref[:80], f"prefill, {bad} in V at 100, H{H} Hkv{Hkv} D{D} {sign}")
        assert not np.isfinite(out[100:].astype(np.float64)).any(), "every later token attends to it"
