"""CPU: which calls of the training operators go through the dispatcher and which run directly.

The kernels are replaced by a recorder (the outputs' values are never looked at): plain eager calls must not
enter the registered op, and every context that looks at operators must see it, as before the direct route.
"""
import contextlib

import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from sorernn_amd import _lib, library, ops


class Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.ops = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.ops.append(str(func))
        return func(*args, **(kwargs or {}))


@pytest.fixture
def launches(monkeypatch):
    calls = []
    monkeypatch.setattr(_lib, "call", lambda name, *a: calls.append(name))
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    entered = []
    for name in ("chunk_fwd", "chunk_bwd", "conv_fwd", "conv_bwd", "l2norm_fwd", "l2norm_bwd", "rms_fwd", "rms_bwd"):
        op = getattr(library, name)
        monkeypatch.setattr(library, name, lambda *a, op=op, name=name: (entered.append(name), op(*a))[1])
    return calls, entered


def _x(*shape, grad=True):
    return torch.randn(*shape).bfloat16().requires_grad_(grad)


def _call(grad=True):
    x, w = _x(1, 8, 16, grad=grad), torch.nn.Parameter(torch.randn(16, 4), requires_grad=grad)
    return x, w, library.conv_fwd_call(x, w, None, None, None, 1, 0, 1, False)[0]


def test_plain_calls_run_directly(launches):
    calls, entered = launches
    _call(grad=False)
    x, w, y = _call()
    torch.autograd.grad(y, [x, w], torch.ones_like(y))
    n = library.l2norm_fwd_call(x.view(8, 16), 1e-12)
    z = library.rms_fwd_call(n, n.detach(), torch.nn.Parameter(torch.ones(16)), None, 1e-6, 1)
    z.sum().backward()
    q, v, g = _x(1, 8, 1, 64), _x(1, 8, 1, 64), torch.zeros(1, 8, 1, requires_grad=True)
    o, fin, states, ws = library.chunk_fwd_call(q, q, v, g, g, None, None, None, None, 0.125, 0, 1, True, True)
    assert o.requires_grad and fin.requires_grad and not states.requires_grad and not ws.requires_grad
    torch.autograd.grad([o, fin], [q, v, g], [torch.ones_like(o), torch.ones_like(fin)])
    assert not entered
    assert calls == ["gdn_causal_conv1d_fwd", "gdn_causal_conv1d_fwd", "gdn_causal_conv1d_bwd", "gdn_l2norm_fwd",
                     "gdn_rms_norm_gated_fwd", "gdn_rms_norm_gated_bwd", "gdn_l2norm_bwd", "gdn_chunk_fwd_train",
                     "gdn_chunk_bwd"]


def test_dispatch_modes_see_the_op(launches):
    with Seen() as seen:
        x, w, y = _call()
        torch.autograd.grad(y, [x, w], torch.ones_like(y))
    assert any("causal_conv1d_fwd" in s for s in seen.ops) and any("causal_conv1d_bwd" in s for s in seen.ops)


def test_transforms_and_subclasses_take_the_op(launches):
    calls, entered = launches

    class Sub(torch.Tensor):
        pass

    x = torch.randn(8, 16).bfloat16()
    library.l2norm_fwd_call(x.as_subclass(Sub), 1e-12)
    assert entered.pop() == "l2norm_fwd" and not entered
    with torch.autograd.forward_ad.dual_level():
        library.l2norm_fwd_call(x, 1e-12)
    assert entered.pop() == "l2norm_fwd" and not entered
    calls.clear()
    y = torch.vmap(lambda t: library.l2norm_fwd_call(t, 1e-12))(x.view(2, 4, 16))  # torch's loop over the op
    assert entered.pop() == "l2norm_fwd" and not entered and calls == ["gdn_l2norm_fwd"] * 2 and y.shape == (2, 4, 16)
    y = torch.fx.experimental.proxy_tensor.make_fx(lambda t: library.l2norm_fwd_call(t, 1e-12))(x)
    assert any("l2norm_fwd" in str(n.target) for n in y.graph.nodes)


def test_saved_tensor_hooks_and_second_derivatives(launches):
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t)[1], lambda t: t):
        x, w, y = _call()
    assert torch.Size([1, 8, 16]) in packed and torch.Size([16, 4]) in packed
    (dx,) = torch.autograd.grad(y, x, torch.ones_like(y), create_graph=True)
    with pytest.raises(RuntimeError, match="autograd formula"):
        dx.sum().backward()


def _chunk(q, v, g):
    return library.chunk_fwd_call(q, q, v, g, g, None, None, None, None, 0.125, 0, 1, False, True)[0]


def _forwards():
    """(name of the backward op, forward of one tensor that requires grad) of every differentiable operator."""
    w, n, g = torch.randn(16, 4), torch.ones(16), torch.zeros(1, 8, 1)
    return [
        ("conv_bwd", lambda x: library.conv_fwd_call(x.view(1, 8, 16), w, None, None, None, 1, 0, 1, False)[0]),
        ("l2norm_bwd", lambda x: library.l2norm_fwd_call(x, 1e-12)),
        ("rms_bwd", lambda x: library.rms_fwd_call(x, None, n, None, 1e-6, 0)),
        ("chunk_bwd", lambda x: _chunk(x.view(1, 2, 1, 64), x.view(1, 2, 1, 64), g[:, :2])),
    ]


@pytest.mark.parametrize("grad_needs_grad", [False, True])
@pytest.mark.parametrize("which", range(4))
def test_second_derivatives_raise(launches, which, grad_needs_grad):
    """A gradient taken with ``create_graph`` depends on the inputs whether or not the incoming one requires grad: a loss
    that holds it next to a differentiable term raises, as no second derivative exists, and is not merely cut short."""
    name, fn = _forwards()[which]
    x, other = _x(8, 16), torch.ones(1, requires_grad=True)
    y = fn(x)
    launches[1].clear()
    (dx,) = torch.autograd.grad(y, x, torch.ones_like(y).requires_grad_(grad_needs_grad), create_graph=True)
    assert launches[1] == [name] and dx.requires_grad
    with pytest.raises(RuntimeError, match="autograd formula"):
        (dx.float().square().sum() + other).backward()


class SeenFunctions(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.ops = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.ops.append(str(func))
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("which", range(4))
def test_function_modes_and_the_profiler_see_the_op(launches, which):
    name, fn = _forwards()[which]
    x = _x(8, 16)
    with SeenFunctions() as seen:
        y = fn(x)
    assert any(s.startswith("sorernn.") for s in seen.ops), seen.ops
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        fn(x).sum().backward()
    ops = {e.name for e in prof.events() if e.name.startswith("sorernn::")}
    assert len(ops) == 2, ops
    launches[1].clear()
    y.sum().backward()
    assert not launches[1]


@pytest.mark.parametrize("context", [None, "vmap", "forward_ad", "function_mode", "profiler"])
def test_range_guard_reads_its_flag_in_every_eager_call(launches, monkeypatch, context):
    """Also where the call takes the registered op because something watches it."""
    monkeypatch.setattr(ops, "_check_cuda", lambda name, *t: t[0].device)
    word = torch.zeros(1, dtype=torch.int32)
    monkeypatch.setattr(ops._range, "_words", {0: (word, word.numpy())})
    monkeypatch.setattr(ops._range, "_device_index", lambda d: 0)
    q, v, g = _x(2, 1, 8, 1, 64, grad=False), _x(1, 8, 1, 64, grad=False), torch.zeros(1, 8, 1)
    fn = lambda t: ops.chunk_gated_delta_rule(t, t, v, g, g)[0].float().sum()  # noqa: E731
    around = {"forward_ad": torch.autograd.forward_ad.dual_level, "function_mode": SeenFunctions,
              "profiler": lambda: torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU])}
    word[0] = 1
    with pytest.warns(RuntimeWarning, match="earlier chunked forward"), around.get(context, contextlib.nullcontext)():
        torch.vmap(fn)(q) if context == "vmap" else fn(q[0])
    assert word.item() == 0


@pytest.mark.parametrize("watched", ["q", "k"])
def test_qk_norm_looks_at_both_tensors(launches, watched):
    calls, entered = launches

    class Sub(torch.Tensor):
        pass

    x = {n: _x(1, 8, 1, 64, grad=False) for n in ("q", "k")}
    ops._l2norm_qk(**x)
    assert calls == ["gdn_qk_l2norm_fwd"] and not entered
    x[watched] = x[watched].as_subclass(Sub)
    ops._l2norm_qk(**x)
    assert entered == ["l2norm_fwd"] * 2


def test_watched_chunk_calls_keep_the_qk_norm_in_the_kernels(launches, monkeypatch):
    calls, _ = launches
    monkeypatch.setattr(ops, "_l2norm_first", lambda *a: True)
    monkeypatch.setattr(ops, "_cus", lambda x: 256)
    x = torch.randn(1, 1000, 16, 128).bfloat16()
    q, k, flags = ops._chunk_qk(x, x, 1, 16, 128, 1000, 7)
    assert flags == 7 & ~_lib.FLAG_QK_L2NORM and calls == ["gdn_qk_l2norm_chunk_fwd"]
    with SeenFunctions():
        q, k, flags = ops._chunk_qk(x, x, 1, 16, 128, 1000, 7)
    assert flags == 7 and q is x and k is x and len(calls) == 1
    asked = []
    monkeypatch.setattr(ops, "_l2norm_first", lambda *a: asked.append(a) or True)
    monkeypatch.setattr(torch.compiler, "is_compiling", lambda: True)
    assert ops._chunk_qk(x, x, 1, 16, 128, 1000, 7)[2] == 7 and not asked  # a compiled graph's guards: none on 1000


@pytest.mark.parametrize("which", range(4))
def test_batched_gradients_loop_over_the_op(launches, which):
    """``is_grads_batched`` and vectorised Jacobians: one launch of the backward per gradient."""
    calls, entered = launches
    name, fn = _forwards()[which]
    x = _x(8, 16)
    y = fn(x)
    calls.clear(), entered.clear()
    (dx,) = torch.autograd.grad(y, x, torch.ones(3, *y.shape, dtype=y.dtype), is_grads_batched=True)
    assert dx.shape == (3, 8, 16) and entered == [name] and len(calls) == 3
    calls.clear()
    jac = torch.autograd.functional.jacobian(lambda t: fn(t).float().sum().view(1), x.detach(), vectorize=True)
    assert jac.shape == (1, 8, 16) and len(calls) == 2


@pytest.mark.parametrize("which", range(4))
def test_jit_traces_hold_the_op(launches, which):
    """A trace that missed the operator would hold its outputs' allocations alone and return uninitialised memory."""
    _, fn = _forwards()[which]
    graph = torch.jit.trace(fn, _x(8, 16, grad=False), check_trace=False).graph
    assert any(n.kind().startswith("sorernn::") for n in graph.nodes()), graph


def test_compiled_call_holds_the_op(launches):
    graphs = []

    def keep(gm, _):
        graphs.append(gm)
        return gm.forward

    torch._dynamo.reset()
    fn = torch.compile(lambda t, w: library.conv_fwd_call(t, w, None, None, None, 1, 0, 1, False)[0], backend=keep, fullgraph=True)
    try:
        fn(torch.randn(1, 8, 16).bfloat16(), torch.randn(16, 4))
    finally:
        torch._dynamo.reset()
    assert any("causal_conv1d_fwd" in str(n.target) for n in graphs[0].graph.nodes)
