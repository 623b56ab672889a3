"""The streaming caches advance in one launch exactly as their Python updates do."""

from __future__ import annotations

import pytest
import torch

from fast_mimi_amd import MimiConfig, MimiConv1dPaddingCache, MimiKVCache, MimiModel
from fast_mimi_amd import _native as nat

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def rt():
    return MimiModel(MimiConfig(num_hidden_layers=1), device=DEV).runtime()


class Slow(MimiConv1dPaddingCache):
    """A subclass: takes its own update()."""


class SlowKV(MimiKVCache):
    """A subclass: takes its own update()."""


@pytest.mark.parametrize("B,C,pad,mode,lengths", [(1, 1, 6, "constant", (1920, 3, 1920)), (3, 64, 2, "constant", (5, 1, 1, 7)),
                                                  (2, 512, 2, "replicate", (2, 1, 4)), (2, 6, 3, "replicate", (1, 1, 9)),
                                                  (1, 8, 0, "constant", (4, 4))])
def test_conv_context(rt, B, C, pad, mode, lengths):
    fast, slow = (c(1, [pad], [mode], [C]) for c in (MimiConv1dPaddingCache, Slow))
    g = torch.Generator().manual_seed(C)
    for n in lengths:
        x = torch.randn(B, n, C, generator=g).to(DEV)
        assert torch.equal(rt._stream_input(x, fast, 0), rt._stream_input(x, slow, 0))
        assert torch.equal(fast.padding_cache[0], slow.padding_cache[0])
        assert fast.padding_cache[0].shape == (B, pad, C)


@pytest.mark.parametrize("B,qd,kd,window,lengths", [(1, 512, 512, 250, (2, 2, 2)), (2, 512, 512, 250, (240, 9, 2, 300)),
                                                    (2, 16, 8, 4, (1, 1, 1, 1, 5)), (1, 6, 6, 3, (4, 2)), (1, 8, 8, 1, (2, 1))])
def test_key_value_cache(rt, B, qd, kd, window, lengths):
    fast, slow = MimiKVCache(0, window), SlowKV(0, window)
    g = torch.Generator().manual_seed(kd)
    for n in lengths:
        q3 = torch.randn(B, n, qd + 2 * kd, generator=g).to(DEV)
        (a, na), (b, nb) = rt._attention_rows(q3, fast, 0, qd, kd), rt._attention_rows(q3, slow, 0, qd, kd)
        assert na == nb and torch.equal(a[:, :, qd:], b[:, :, qd:]) and torch.equal(a[:, na:], b[:, nb:])
        for f, s in ((fast.key_cache, slow.key_cache), (fast.value_cache, slow.value_cache)):
            assert torch.equal(f[0], s[0])
        assert fast.get_seq_length() == slow.get_seq_length()


@pytest.mark.parametrize("B,nh,nkv,lengths", [(1, 8, 8, (2, 2, 240, 17, 2)), (2, 8, 2, (15, 16, 300, 1)), (1, 2, 1, (511, 33)),
                                              (17, 8, 8, (3, 2)), (3, 4, 4, (250, 600, 4))])
def test_attention_advances_the_cache(rt, B, nh, nkv, lengths):
    """One launch gives the attention's and the caches' bits of the two before it."""
    window = rt.config.sliding_window
    one, two = MimiKVCache(0, window), MimiKVCache(0, window)
    qd, kd = 64 * nh, 64 * nkv
    g = torch.Generator().manual_seed(B + nh)
    for n in lengths:
        q3 = torch.randn(B, n, qd + 2 * kd, generator=g).to(DEV)
        a, b = (torch.full((B * n, qd), float("nan"), device=DEV) for _ in range(2))
        if not rt._attend_stream(q3, one, 0, nh, nkv, 64, a):
            comb, past = rt._attention_rows(q3, one, 0, qd, kd)
            rt._call("fm_window_attention_rows", comb, qd + 2 * kd, 0, qd, qd + kd, None, None, B, past + n, past, nh,
                     nkv, 64, window, 0.125, a, qd)
        else:
            assert n < 512
        comb, past = rt._attention_rows(q3, two, 0, qd, kd)
        rt._call("fm_window_attention_rows", comb, qd + 2 * kd, 0, qd, qd + kd, None, None, B, past + n, past, nh, nkv,
                 64, window, 0.125, b, qd)
        assert torch.equal(a, b)
        assert torch.equal(one.key_cache[0], two.key_cache[0]) and torch.equal(one.value_cache[0], two.value_cache[0])
        assert one.get_seq_length() == two.get_seq_length()


def test_foreign_cache_tensors(rt):
    """Strided context and key tensors, as a caller may put there, still serve;
    a context of another shape is refused as before."""
    g = torch.Generator().manual_seed(0)
    x = torch.randn(2, 4, 8, generator=g).to(DEV)
    cache = MimiConv1dPaddingCache(1, [2], ["constant"], [8])
    ctx = torch.randn(2, 8, 2, generator=g).to(DEV).transpose(1, 2)
    cache.padding_cache[0] = ctx
    assert torch.equal(rt._stream_input(x, cache, 0), torch.cat((ctx, x), 1))
    cache.padding_cache[0] = torch.zeros(1, 2, 8, device=DEV)
    with pytest.raises(RuntimeError):
        rt._stream_input(x, cache, 0)
    kv = MimiKVCache(1, 5)
    kv.key_cache[0] = kv.value_cache[0] = torch.randn(2, 4, 3, generator=g).to(DEV).transpose(1, 2)
    comb, n = rt._attention_rows(torch.randn(2, 1, 12, generator=g).to(DEV), kv, 0, 4, 4)
    assert n == 3 and comb.shape == (2, 4, 12) and kv.key_cache[0].shape == (2, 4, 4)


def test_rejects():
    t = torch.zeros(64, device=DEV).data_ptr()
    for args in ((t, t, 1, 0, 4, 4, 0, t, t), (t, t, 1, 2, 0, 4, 0, t, t), (t, None, 1, 2, 4, 4, 0, t, t)):
        with pytest.raises(nat.NativeError, match="bad argument"):
            nat.call("fm_stream_append", *args, 0)
    for args in ((t, 4, 4, 1, 2, None, None, 1, 1, t, t, t), (t, 4, 4, 1, 2, t, t, 1, 4, t, t, t),
                 (t, 4, 4, 1, 2, t, t, 1, 1, t, None, t)):
        with pytest.raises(nat.NativeError, match="bad argument"):
            nat.call("fm_kv_append", *args, 0)
