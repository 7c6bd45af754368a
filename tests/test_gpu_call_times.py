"""Calls whose route is chosen by their sizes, against another route to the
same result: the chosen one must not cost a multiple of the other. Times are
the best of several replays of a graph of equal calls, so the host's part is
not in them, and the margins are far above what two runs differ by."""

import numpy as np
import pytest

from swiftllm_amd import paged_attention as pa
from swiftllm_amd._hip import DeviceArray, Event, Graph, Stream

pytestmark = pytest.mark.gpu


def best_us(call, calls=20, replays=8):
    """Microseconds per call(stream)."""
    stream = Stream()
    call(stream)  # code objects are loaded before the capture
    stream.synchronize()
    graph = Graph(stream, lambda: [call(stream) for _ in range(calls)])
    best = float("inf")
    for _ in range(replays):
        a, b = Event(), Event()
        a.record(stream)
        graph.launch(stream)
        b.record(stream)
        b.synchronize()
        best = min(best, a.elapsed_ms(b) * 1e3 / calls)
    return best


@pytest.mark.parametrize("S,L,H,Hkv,D", [(1000, 64, 8, 8, 64), (300, 16, 32, 8, 128)])
def test_many_short_prompts(dev, S, L, H, Hkv, D):
    """A positive scale may take the kernel with shared stages, a negative one
    takes the per-wave kernel: on many prompts of a few tokens a positive one
    costs no more (at most 64 tokens each, 8/8 x 64: 60 us against 46 where
    such calls shared their stages)."""
    rng = np.random.default_rng(S + L)
    lens = rng.integers(1, L + 1, size=S).astype(np.int32)
    lens[0] = L
    nb = (lens + 15) // 16
    first = np.cumsum(nb) - nb
    slots = np.concatenate([16 * f + np.arange(n) for f, n in zip(first, lens)]).astype(np.int32)
    T, NB = int(lens.sum()), int(nb.sum())
    def arr(*shape):
        return DeviceArray.from_numpy((rng.standard_normal(shape) * 0.5).astype(np.float16))
    q, kc, vc = arr(T, H, D), arr(NB, Hkv, D, 16), arr(NB, Hkv, D, 16)
    sm, ctx, out = DeviceArray.from_numpy(slots), DeviceArray.from_numpy(lens), DeviceArray((T, H, D), np.float16)
    us = [best_us(lambda stream: pa.launch_paged_prefill(out, q, kc, vc, sm, ctx, sign / np.sqrt(D), S, H, Hkv, D,
                                                         16, L, num_blocks=NB, stream=stream))
          for sign in (1, -1)]
    assert us[0] < 1.15 * us[1], f"{us[0]:.1f} us, per wave {us[1]:.1f} us"


@pytest.mark.parametrize("Hkv,D", [(2, 128), (1, 128)])
def test_cache_write_of_short_runs(dev, Hkv, D):
    """Two new tokens for each of 257 sequences into a layer of one or two kv
    heads. Caches 4 bytes past an 8-byte boundary take the kernel
    that writes token by token, and the calls that find runs cost no more than
    it (9.8 and 6.8 us against 6.2 and 4.7 with windows of 16 tokens)."""
    rng = np.random.default_rng(Hkv)
    T, NB = 514, 600
    blocks = rng.permutation(NB)[:T // 2]
    slots = (16 * np.repeat(blocks, 2) + np.tile([4, 5], T // 2)).astype(np.int32)
    key, value = (DeviceArray.from_numpy(rng.standard_normal((T, Hkv, D)).astype(np.float16)) for _ in range(2))
    kc, vc = (DeviceArray((NB * Hkv * D * 16 + 8,), np.float16) for _ in range(2))
    sm = DeviceArray.from_numpy(slots)
    us = [best_us(lambda stream: pa.launch_reshape_and_cache(key, value, kc.ptr + shift, vc.ptr + shift, sm, T, Hkv,
                                                             D, 16, num_blocks=NB, stream=stream))
          for shift in (0, 4)]
    assert us[0] < 1.2 * us[1], f"{us[0]:.2f} us, token by token {us[1]:.2f} us"


class _Decode:
    """A decode batch whose contexts take random blocks of a small pool."""

    def __init__(self, lens, H, Hkv, D, table_blocks):
        rng = np.random.default_rng(len(lens))
        self.lens = np.asarray(lens, np.int32)
        S, NB = len(lens), 4096
        self.shape = (S, H, Hkv, D, 16, table_blocks)
        self.nb, self.scale = NB, 1.0 / np.sqrt(D)
        fill = (rng.standard_normal((NB * Hkv * D * 16,)) * 0.5).astype(np.float16)
        self.kc, self.vc = DeviceArray.from_numpy(fill), DeviceArray.from_numpy(fill[::-1].copy())
        self.q = DeviceArray.from_numpy(rng.standard_normal((S, H, D)).astype(np.float16))
        self.bt = DeviceArray.from_numpy(rng.integers(0, NB, (S, table_blocks)).astype(np.int32))
        self.ctx = DeviceArray.from_numpy(self.lens)
        self.out = DeviceArray((S, H, D), np.float16)

    def v1(self, stream):
        pa.paged_attention_v1(self.out, self.q, self.kc, self.vc, self.bt, self.ctx, self.scale, *self.shape,
                              num_blocks=self.nb, stream=stream)

    def v2(self, partition):
        ws = pa.workspace(pa.paged_attention_v2_workspace_size(*self.shape, partition))
        return lambda stream: pa.paged_attention_v2(self.out, ws, self.q, self.kc, self.vc, self.bt, self.ctx,
                                                    self.scale, *self.shape, partition, num_blocks=self.nb,
                                                    stream=stream)


@pytest.mark.parametrize("S,long", [(64, 2500), (96, 3500)])
@pytest.mark.parametrize("partition", [512, 0])
def test_one_long_context_among_short_ones_is_split(dev, S, long, partition):
    """All contexts of 32 tokens but one: a split call spreads the long one over
    workgroups, where the single pass walks it in one per kv head (64 with one
    of 2500 tokens 32 us and split 15, 96 with one of 3500 44 and 19)."""
    d = _Decode([32] * (S - 1) + [long], 32, 8, 128, (long + 15) // 16)
    split, single = best_us(d.v2(partition)), best_us(d.v1)
    assert split < 0.75 * single, f"{split:.1f} us, single pass {single:.1f} us"


@pytest.mark.parametrize("S,H,Hkv,D", [(256, 32, 8, 128), (256, 8, 8, 64), (1024, 8, 8, 64)])
def test_single_pass_of_short_contexts_under_wide_tables(dev, S, H, Hkv, D):
    """The table's width is what a program allocates, not what a batch needs:
    contexts of 16-128 tokens cost about the same under tables for 8192 (they
    went through a list that each workgroup builds: 27 us against 17, 17.5
    against 9.3, 65 against 28)."""
    lens = np.random.default_rng(S).integers(16, 129, size=S)
    us = [best_us(_Decode(lens, H, Hkv, D, blocks).v1) for blocks in (512, 8)]
    assert us[0] < 1.5 * us[1], f"{us[0]:.1f} us, tables of 8 blocks {us[1]:.1f} us"


@pytest.mark.parametrize("S", [64, 96])
@pytest.mark.parametrize("partition", [512, 0])
def test_split_of_short_contexts_under_wide_tables(dev, S, partition):
    """Teams do not cut contexts of 16-128 tokens: a split call takes them whole
    and costs one empty kernel more than the single pass (96 of them 19.5 us
    cut, 11.7 whole, single pass 10.9)."""
    lens = np.random.default_rng(S).integers(16, 129, size=S)
    d = _Decode(lens, 32, 8, 128, 512)
    split, single = best_us(d.v2(partition)), best_us(d.v1)
    assert split < 1.5 * single, f"{split:.1f} us, single pass {single:.1f} us"
