"""The two routes of an op (``ops._Op``): the direct call of plain eager tensors
and the dispatcher.  On the CPU, with ops made of torch arithmetic: which calls
take which route, and that both give the same results, gradients, saved-tensor
hooks and version counts.  The public functions and a layer are traced with fake
GPU tensors into one graph (``torch.compile(fullgraph=True)``)."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils._python_dispatch import TorchDispatchMode

from mogt_amd import ops

CALLS = []


def _scale_impl(x: torch.Tensor, y: torch.Tensor, k: float) -> tuple[torch.Tensor, torch.Tensor]:
    CALLS.append(torch.is_grad_enabled() and (x.requires_grad or y.requires_grad))
    return x * y * k, x + k


_scale = ops._op("mogt::route_test_scale")(_scale_impl)


@_scale.register_fake
def _(x, y, k):
    return torch.empty_like(x), torch.empty_like(x)


def _scale_setup(ctx, inputs, output):
    x, y, k = inputs
    ctx.save_for_backward(x, y, output[0])
    ctx.k = k
    ctx.set_materialize_grads(False)


def _scale_backward(ctx, g0, g1):
    x, y, _ = ctx.saved_tensors
    gx = None if g0 is None else g0 * y * ctx.k
    if g1 is not None:
        gx = g1 if gx is None else gx + g1
    return gx, None if g0 is None else g0 * x * ctx.k, None


_scale.register_autograd(_scale_backward, _scale_setup)


def _fill_impl(out: torch.Tensor, v: float) -> None:
    with torch.no_grad():
        out.detach().view(-1)[:] = v


_fill = ops._op("mogt::route_test_fill_", mutates=("out",))(_fill_impl)


class _Spy:
    """Counts the calls that go through the dispatcher."""

    def __init__(self, monkeypatch, op):
        self.n = 0
        through = op.dispatched

        def spy(*args):
            self.n += 1
            return through(*args)

        monkeypatch.setattr(op, "dispatched", spy)


class _Mode(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("parameter", [False, True])
def test_plain_calls_run_directly_with_the_dispatchers_results(monkeypatch, parameter):
    spy = _Spy(monkeypatch, _scale)
    x, y = torch.randn(5), torch.randn(5)
    if parameter:
        y = torch.nn.Parameter(y)
    with torch.no_grad():
        a, b = _scale(x, y, 2.0)
    assert spy.n == 0 and torch.equal(a, x * y * 2.0) and torch.equal(b, x + 2.0)
    for need in ((True, False), (False, True), (True, True)):
        grads = []
        for run in (_scale, torch.ops.mogt.route_test_scale):
            xs, ys = x.detach().clone().requires_grad_(need[0]), y.detach().clone().requires_grad_(need[1])
            o0, o1 = run(xs, ys, 2.0)
            assert o0.requires_grad and o1.requires_grad
            (o0.sum() + (3 * o1).sum()).backward()
            grads.append((xs.grad, ys.grad))
            xs.grad = ys.grad = None
            _scale(xs, ys, 2.0)[0].sum().backward()   # the second output unused
            grads[-1] += (xs.grad, ys.grad)
        for g, r in zip(*grads):
            assert (g is None) == (r is None) and (g is None or torch.equal(g, r))
    assert spy.n == 0 and not any(CALLS)   # no implementation ran with autograd recording


def test_special_calls_go_through_the_dispatcher(monkeypatch):
    spy = _Spy(monkeypatch, _scale)
    x, y = torch.randn(4), torch.randn(4)

    def took(n):
        assert spy.n == n, (spy.n, n)

    with _Mode():
        _scale(x, y, 1.0)
    took(1)
    with FakeTensorMode() as fm:
        f = fm.from_tensor(x)
        assert _scale(f, f, 1.0)[0].shape == x.shape
    took(2)
    g = make_fx(lambda u, v: _scale(u, v, 1.0)[0])(x, y)
    took(3)
    assert any("route_test_scale" in str(n.target) for n in g.graph.nodes)
    with torch.device("cpu"):        # a function mode
        _scale(x, y, 1.0)
    took(4)
    with torch.autograd.forward_ad.dual_level():
        _scale(x, y, 1.0)
    took(5)
    neg = torch.imag(torch.complex(x, y).conj())
    assert neg.is_neg()
    assert torch.equal(_scale(neg, y, 1.0)[0], -y * y)
    took(6)

    class Sub(torch.Tensor):
        pass

    _scale(x.as_subclass(Sub), y, 1.0)
    took(7)
    try:
        torch.vmap(lambda u: _scale(u, u, 1.0)[0])(torch.randn(2, 3))
    except Exception:                # no batching rule: the dispatcher's own answer
        pass
    took(8)
    _scale(x, y, 1.0)
    took(8)


def test_saved_tensor_hooks_see_the_direct_route():
    x, y = torch.randn(4, requires_grad=True), torch.randn(4, requires_grad=True)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t) or t.clone(), lambda t: t):
        o, _ = _scale(x, y, 2.0)
    assert len(seen) == 3
    o.sum().backward()
    assert torch.equal(x.grad, 2 * y.detach()) and torch.equal(y.grad, 2 * x.detach())


def test_written_arguments_count_a_version(monkeypatch):
    spy = _Spy(monkeypatch, _fill)
    t = torch.zeros(3)
    before = t._version
    _fill(t, 4.0)
    assert spy.n == 0 and t._version > before and float(t[0]) == 4.0
    with torch.inference_mode():
        u = torch.zeros(3)
        _fill(u, 5.0)
    assert float(u[2]) == 5.0
    # a tensor autograd saved and the op overwrote is refused in the backward
    a = torch.randn(3, requires_grad=True)
    s = torch.ones(3)
    z = (a * s).sum()
    _fill(s, 2.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        z.backward()


class _Traced(Exception):
    pass


def _trace(fn, *args):
    """The one graph torch.compile makes of the call, traced and not run."""
    graphs = []

    def backend(gm, inputs):
        graphs.append(gm)

        def run(*a):
            raise _Traced

        return run

    torch._dynamo.reset()
    with pytest.raises(_Traced):
        torch.compile(fn, fullgraph=True, backend=backend)(*args)
    (graph,) = graphs
    return "".join(m.code for m in graph.modules() if isinstance(m, torch.fx.GraphModule))


def _fake(*shape, dtype=torch.float32, grad=False):
    with _FAKE:
        return torch.empty(*shape, dtype=dtype, device="cuda").requires_grad_(grad)


_FAKE = FakeTensorMode()


def test_profiled_functions_trace_into_one_graph():
    """The hybrid scan with gradients and a layer in training, whose parts sit in
    profiler ranges."""
    from mogt_amd import model_mogt, triton_scan

    code = _trace(triton_scan.triton_affine_scan_hybrid, _fake(1, 100, 16, 16, grad=True), _fake(1, 100, 16, 48, grad=True))
    assert "affine_scan_carry" in code
    for connection in ("identity", "matrix_exp"):
        with _FAKE, torch.device("cuda"):
            block = model_mogt.MOGTBlock(d_model=128, r=16, ffn_hidden=256)
        block.connection_impl, block.scan_impl = connection, "triton_hybrid"
        code = _trace(lambda x: block(x), _fake(1, 64, 128))
        assert ("diag_scan" if connection == "identity" else "connection_map") in code


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_chunked_loss_traces_into_one_graph(dtype):
    """The tied-head loss with gradients at a size whose products take the split
    form."""
    from mogt_amd import chunked_lm_loss as cl

    code = _trace(lambda h, w, labels: cl.chunked_linear_cross_entropy(h, w, labels, chunk_size=1024),
                  _fake(1, 2000, 768, dtype=dtype, grad=True), _fake(32000, 768, grad=True),
                  _fake(1, 2000, dtype=torch.int64))
    assert "split_head_loss" in code and "split_gemm_" in code
