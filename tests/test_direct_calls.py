"""ops.call takes the C function directly only when nothing observes operator
calls, and a streamed RoPE table is a slice of a longer one (CPU only)."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from fast_mimi_amd import MimiConfig, MimiModel, ops
from fast_mimi_amd.runtime import MimiRuntime, _plain, rope_tables


def test_observers_keep_the_operator_path():
    seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class FunctionMode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    def look(x):
        seen.append(ops._observed())
        return x * 2

    x = torch.ones(3)
    assert not ops._observed()
    with Mode():
        look(x)
    with FunctionMode():
        look(x)
    torch.vmap(look)(x)
    torch.func.jvp(look, (x,), (x,))
    torch.func.grad(lambda v: look(v).sum())(x)
    torch.jit.trace(look, (x,), check_trace=False)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]):
        look(x)
    assert len(seen) >= 7 and all(seen)
    assert not ops._observed()


def test_compiled_in_one_graph():
    """torch.compile traces ops.call as the operator, without a graph break."""
    graphs = []

    def keep(gm, inputs):
        graphs.append(gm)
        return lambda *args: args[-1:]  # (the operator itself needs a GPU)

    def body(src, dst):
        ops.call("fm_copy_buffers", src, dst, 16, None, None, 0)
        return dst + 1

    torch._dynamo.reset()
    torch.compile(body, backend=keep, fullgraph=True)(torch.ones(4), torch.zeros(4))
    assert len(graphs) == 1
    assert any("copy_buffers" in str(n.target) for n in graphs[0].graph.nodes if n.op == "call_function")


def test_lazily_negated_inputs_are_resolved():
    """A tensor with the negative bit holds other values than its memory; the
    operators resolved it, direct calls pass its address."""
    x = torch.arange(4.0).view(1, 1, 4)
    neg = torch._neg_view(x)
    got = MimiModel._on_device(SimpleNamespace(device=x.device), neg, torch.float32)
    assert not got.is_neg() and torch.equal(got, -x) and got.data_ptr() != x.data_ptr()
    assert MimiModel._on_device(SimpleNamespace(device=x.device), x, torch.float32).data_ptr() == x.data_ptr()
    assert _plain(x, x, (1, 1, 4)) and not _plain(neg, x, (1, 1, 4))


def test_pointer_arguments_follow_the_schema():
    for entry, spec in ops.SPECS.items():
        kinds = [item.split(":")[0] for item in spec.split()]
        assert ops._POINTERS[entry] == tuple(i for i, k in enumerate(kinds) if k in ("in", "out", "res"))


def test_rope_table_prefixes():
    whole = rope_tables(MimiConfig(), 2048)
    for n in (1, 2, 3, 7, 100, 251, 777, 2047):
        for a, b in zip(whole, rope_tables(MimiConfig(), n)):
            assert torch.equal(a[:n], b)


def test_prepared_stream_tables_serve_a_capture(monkeypatch):
    """While a graph is captured no table can be uploaded: a streamed chunk
    takes the one prepare() made for its end position."""
    rt = MimiRuntime.__new__(MimiRuntime)
    rt.config, rt.device, rt._rope, rt._stream_tabs = MimiConfig(), torch.device("cpu"), {}, []
    capturing = [False]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    rt.prepare(700)
    capturing[0] = True
    whole = rope_tables(rt.config, 700)
    for got, want in zip(rt._stream_rope(698, 2), whole):
        assert torch.equal(got, want[698:])
    with pytest.raises(RuntimeError, match="prepared"):
        rt._stream_rope(699, 2)
    capturing[0] = False
    rt._stream_rope(699, 2)
    capturing[0] = True
    assert rt._stream_rope(1000, 24)[0].shape == (24, 64)
    with pytest.raises(RuntimeError, match="prepared"):
        rt._stream_rope(1000, 25)
