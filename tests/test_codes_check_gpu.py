"""decode queues its work behind the range check and still refuses bad codes."""

from __future__ import annotations

import threading

import pytest
import torch

from fast_mimi_amd import MimiConfig, MimiKVCache, MimiModel
from fast_mimi_amd import _native as nat

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def model():
    return MimiModel(MimiConfig(num_hidden_layers=2), device=DEV)


def codes(seed, t=13, b=1):
    return torch.randint(0, 2048, (b, 8, t), generator=torch.Generator().manual_seed(seed)).to(DEV)


@pytest.mark.parametrize("n,at,value,bad", [(1, 0, 2048, 1), (1, 0, 2047, 0), (1000, 999, -1, 1), (300_000, 123_457, 1 << 40, 1),
                                            (300_001, 300_000, -(1 << 63), 1), (300_000, 0, 0, 0), (0, 0, 0, 0)])
def test_flag(n, at, value, bad):
    c = torch.randint(0, 2048, (n,), device=DEV)
    if n:
        c[at] = value
    flag = torch.zeros(1, dtype=torch.int32, pin_memory=True)
    nat.call("fm_codes_check", c.data_ptr() if n else flag.data_ptr(), n, 2048, flag.data_ptr(),
             torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert flag.item() == bad


@pytest.mark.parametrize("graphs", [True, False])
def test_bad_codes_refused_and_state_kept(model, graphs):
    model.use_graphs = graphs
    good = codes(1)
    want = model.decode(good).audio_values
    worse = good.clone()
    worse[0, 7, 12] = 2048
    for bad in (worse, codes(2, t=9) - 2048):
        with pytest.raises(IndexError):
            model.decode(bad)
    assert torch.equal(model.decode(good).audio_values, want)
    # A cache the refused call was given is as it was.
    kv = MimiKVCache(2, 250)
    ref = [model.decode(codes(s, t=2), decoder_past_key_values=kv).audio_values for s in (3, 4)]
    kv = MimiKVCache(2)
    first = model.decode(codes(3, t=2), decoder_past_key_values=kv).audio_values
    before = (list(kv.key_cache), list(kv.value_cache), kv.get_seq_length(), kv.sliding_window)
    with pytest.raises(IndexError):
        model.decode(codes(4, t=2) + 2048, decoder_past_key_values=kv)
    assert (kv.get_seq_length(), kv.sliding_window) == before[2:]
    assert all(a is b for a, b in zip(kv.key_cache + kv.value_cache, before[0] + before[1]))
    second = model.decode(codes(4, t=2), decoder_past_key_values=kv).audio_values
    assert torch.equal(first, ref[0]) and torch.equal(second, ref[1])
    model.use_graphs = True


def test_bad_codes_of_a_new_shape_build_nothing(model):
    """A refused call of a shape seen for the first time captures no graph
    (each would keep a memory pool)."""
    before = set(model._graphs)
    for t in (17, 19):
        with pytest.raises(IndexError):
            model.decode(codes(6, t=t) + 2048)
    assert set(model._graphs) == before
    model.decode(codes(6, t=17))
    assert len(model._graphs) == len(before) + 1


def test_refused_call_keeps_the_cache_lists(model):
    """The lists a caller holds of a cache stay the cache's own."""
    kv = MimiKVCache(2)
    model.decode(codes(3, t=2), decoder_past_key_values=kv)
    keys, values, lengths = kv.key_cache, kv.value_cache, kv._cumulative_lengths
    with pytest.raises(IndexError):
        model.decode(codes(4, t=2) + 2048, decoder_past_key_values=kv)
    assert kv.key_cache is keys and kv.value_cache is values and kv._cumulative_lengths is lengths
    assert kv.get_seq_length() == 4 and keys[0].shape[1] == 4


def test_foreign_cache_is_not_touched(model):
    class Mine(MimiKVCache):
        pass

    kv = Mine(2, 250)
    with pytest.raises(IndexError):
        model.decode(codes(5, t=2) + 2048, decoder_past_key_values=kv)
    assert kv.get_seq_length() == 0 and kv.key_cache == [None, None]


def test_threads(model):
    """Good and bad calls from several threads."""
    want = {s: model.decode(codes(s)).audio_values for s in range(4)}
    torch.cuda.synchronize()
    wrong = []

    def work(s):
        c = codes(s)
        for i in range(6):
            try:
                out = model.decode(c if i % 2 == 0 else c + 2048).audio_values
                if i % 2 or not torch.equal(out, want[s]):
                    wrong.append((s, i))
            except IndexError:
                if i % 2 == 0:
                    wrong.append((s, i))

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    assert 1 <= len(model._check_flags) <= 5
