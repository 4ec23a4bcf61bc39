"""Rules that send a projection from the library to a hand-written kernel, on the CPU: every call that only the library
can answer is left to it.  The kernels' entry points are replaced by one that says so instead of launching."""
import pytest
import torch
import torch.nn.functional as F

from minivllm_amd import ops
from minivllm_amd.ops import hip, torch_ref

BF = torch.bfloat16


class Launched(Exception):
    pass


@pytest.fixture(autouse=True)
def no_gpu(monkeypatch):
    def launch(*a):
        raise Launched
    monkeypatch.setattr(ops, "_on_gpu", torch.is_tensor)
    monkeypatch.setattr(hip, "_stream", lambda: 0)
    for name in ("_skinny", "_skinny_splitk", "_skinny_norm", "_mid", "_mid_reduce", "_splitk_norm", "_big"):
        monkeypatch.setattr(hip, name, launch)
    for name in ("rms_norm", "add_rms_norm", "silu_and_mul"):
        monkeypatch.setattr(hip, name, getattr(torch_ref, name))
    for name in ("_SKINNY_CHOICE", "_MID_CHOICE", "_BIG_CHOICE"):
        monkeypatch.setattr(hip, name, {})


def _linear(x, w, b):
    return ops.linear(x, w, b, to_norm=True)


# entry point, rows, output columns: each a call that a rule sends to a kernel
CALLS = {"narrow to norm": (_linear, 4, 1024), "several row tiles": (_linear, 300, 1024),
         "several row tiles, SwiGLU": (ops.swiglu_linear, 300, 2048)}


def _operands(rows, n):
    torch.manual_seed(rows + n)
    return torch.randn(rows, 1024).to(BF), (torch.randn(n, 1024) / 32).to(BF)


def _by_library(call, x, w, b):
    """The call is answered without a kernel, as the library answers it."""
    got, want = call(x, w, b), F.linear(x, w, b)
    torch.testing.assert_close(got, want if got.shape == want.shape else torch_ref.silu_and_mul(want))
    return got


@pytest.mark.parametrize("call,rows,n", CALLS.values(), ids=CALLS)
def test_biases(call, rows, n):
    """A kernel reads as many bias values as there are columns, next to each other, in the weight's type."""
    x, w = _operands(rows, n)
    b = torch.randn(2 * n + 1).to(BF)
    for plain in (None, b[:n]):
        with pytest.raises(Launched):
            call(x, w, plain)
    for other in (b[:1], b[:n].view(1, n), torch.randn(rows, n).to(BF), b[:1].expand(n), b[:2 * n:2], b[1:n + 1]):
        _by_library(call, x, w, other)
    for refused in (torch.randn(n), b[:n - 1]):
        with pytest.raises(RuntimeError):
            call(x, w, refused)


def _norm_linear(x, w, b, slices=0, swiglu=False):
    """Residual add + norm + projection, from a tensor or from the slices of the projection before it."""
    ones, rows = torch.ones(1024, dtype=BF), torch.zeros_like(x)
    if slices:
        x = hip.SplitKPartials(x.detach()[None].float(), None, BF)
    return ops.norm_linear(x, rows, ones, 1e-6, w, b, swiglu, gamma_folded=True)[0]


# entry point, rows: each a call that runs as one kernel
NORMED = {"1 row": (_norm_linear, 1), "4 rows": (_norm_linear, 4), "16 rows": (_norm_linear, 16),
          "slices": (lambda x, w, b: _norm_linear(x, w, b, slices=1), 4),
          "SwiGLU": (lambda x, w, b: _norm_linear(x, w, b, swiglu=True), 4),
          "slices, SwiGLU": (lambda x, w, b: _norm_linear(x, w, b, 1, True), 3)}


@pytest.mark.parametrize("call,rows", NORMED.values(), ids=NORMED)
def test_biases_behind_a_norm(monkeypatch, call, rows):
    """As ``test_biases``; what is not for the one kernel is what the norm and the library's projection give."""
    monkeypatch.setattr(hip.SplitKPartials, "add_rms_norm",
                        lambda p, r, g, eps: torch_ref.add_rms_norm(p.ws.sum(0).to(p.dtype), r, g, eps))
    n = 2048
    x, w = _operands(rows, n)
    b = torch.randn(2 * n + 1).to(BF)
    normed = lambda x, w, b: call(x.clone(), w, b)
    library = lambda x, w, b: F.linear(torch_ref.rms_norm(x, torch.ones(1024, dtype=BF), 1e-6), w, b)
    for plain in (None, b[:n], b[1:n + 1]):
        with pytest.raises(Launched):
            normed(x, w, plain)
    for other in (b[:1], b[:n].view(1, n), torch.randn(rows, n).to(BF), b[:1].expand(n), b[:2 * n:2]):
        got, want = normed(x, w, other), library(x, w, other)
        torch.testing.assert_close(got, want if got.shape == want.shape else torch_ref.silu_and_mul(want))
    for refused in (torch.randn(n), b[:n - 1]):
        with pytest.raises(RuntimeError):
            normed(x, w, refused)
    wg = w.clone().requires_grad_()
    normed(x, wg, b[:n]).float().sum().backward()
    assert wg.grad is not None
    with torch.no_grad(), pytest.raises(Launched):
        normed(x, wg, b[:n])


def _transforms(call):
    """name -> (function of x, w, b, what a call under that transform gives)."""
    fw = torch.autograd.forward_ad

    def bias_gradient(x, w, b):
        b = b.clone().requires_grad_()
        call(x, w, b).float().sum().backward()
        return b.grad

    def tangent(of):
        def f(*args):
            with fw.dual_level():
                args = list(args)
                args[of] = fw.make_dual(args[of], torch.ones_like(args[of]))
                return fw.unpack_dual(call(*args)).tangent
        return f

    def other_types(x, w, b):
        from torch._subclasses import FakeTensorMode
        with FakeTensorMode() as mode:
            fake = [mode.from_tensor(t) for t in (x, w, b)]
        return torch.empty(call(*fake).shape)                # (out of the mode: the tensors carry it)

    def counted(x, w, b):
        from torch.utils.flop_counter import FlopCounterMode
        with FlopCounterMode(display=False) as c:
            call(x, w, b)
        return torch.tensor(c.get_total_flops())

    def autocast(x, w, b):
        torch.set_autocast_enabled("cuda", True)
        try:
            return call(x, w, b)
        finally:
            torch.set_autocast_enabled("cuda", False)

    return {"gradient of the bias": bias_gradient, "tangent of x": tangent(0), "tangent of the weight": tangent(1),
            "tangent of the bias": tangent(2), "vmap over weights": lambda x, w, b: torch.func.vmap(
                lambda ww: call(x, ww, b))(torch.stack([w, -w])),
            "jvp": lambda x, w, b: torch.func.jvp(lambda t: call(x, w, t), (b,), (torch.ones_like(b),))[1],
            "jit trace": lambda x, w, b: torch.jit.trace(call, (x, w, b), check_trace=False)(2 * x, w, b),
            "fx trace": lambda x, w, b: torch.fx.experimental.proxy_tensor.make_fx(call)(x, w, b)(2 * x, w, b),
            "compiled": lambda *a: torch.compile(call, backend="eager", fullgraph=True)(*a),
            "fake tensors": other_types, "counted": counted, "autocast": autocast}


@pytest.mark.filterwarnings("ignore")                        # (of the tracers)
@pytest.mark.parametrize("call,rows,n", [CALLS["narrow to norm"], CALLS["several row tiles"]])
@pytest.mark.parametrize("name", list(_transforms(None)))
def test_transforms(call, rows, n, name):
    """Calls of which more than the values is wanted: as the library's projection gives it."""
    import torch.fx.experimental.proxy_tensor                # noqa: F401
    x, w = _operands(rows, n)
    b = torch.randn(n).to(BF)
    got, want = (_transforms(c)[name](x, w, b) for c in (call, F.linear))
    assert got is not None
    torch.testing.assert_close(got, want) if name != "fake tensors" else None
    assert got.shape == want.shape
    with pytest.raises(Launched):                            # (and nothing is left switched off)
        call(x, w, b)


@pytest.mark.parametrize("rows", [2, 4])
@pytest.mark.parametrize("slices", [0, 1])
def test_transforms_behind_a_norm(monkeypatch, rows, slices):
    monkeypatch.setattr(hip.SplitKPartials, "add_rms_norm",
                        lambda p, r, g, eps: torch_ref.add_rms_norm(p.ws.sum(0).to(p.dtype), r, g, eps))
    x, w = _operands(rows, 2048)
    b = torch.randn(2048).to(BF)
    call = lambda ww, bb: _norm_linear(x.clone(), ww, bb, slices)
    bg = b.clone().requires_grad_()
    call(w, bg).float().sum().backward()
    assert torch.equal(bg.grad, torch.full_like(b, rows))
    for wrt in (0, 1):
        with torch.autograd.forward_ad.dual_level():
            args = [w, b]
            args[wrt] = torch.autograd.forward_ad.make_dual(args[wrt], torch.ones_like(args[wrt]))
            assert torch.autograd.forward_ad.unpack_dual(call(*args)).tangent is not None
    assert torch.func.vmap(lambda ww: call(ww, b))(torch.stack([w, -w])).shape == (2, rows, 2048)
    with pytest.raises(Launched):
        call(w, b)


@pytest.mark.parametrize("rows", [1, 4, 16, 40, 300])
@pytest.mark.parametrize("call,n,kind", [(ops.linear, 1024, False), (_linear, 1024, "norm"), (ops.swiglu_linear, 2048, True)],
                         ids=["plain", "to norm", "SwiGLU"])
def test_biases_of_measured_projections(monkeypatch, rows, call, n, kind):
    """The same where the start-up timing chose a kernel for the shape."""
    for b in (1, 8, 16):
        monkeypatch.setitem(hip._SKINNY_CHOICE, (b, n, 1024, kind), True if kind != "norm" else 2)
    monkeypatch.setitem(hip._MID_CHOICE, (64, n, 1024, kind), (64, 2, True))
    monkeypatch.setitem(hip._BIG_CHOICE, (512, n, 1024, kind is True), True)
    x, w = _operands(rows, n)
    b = torch.randn(2 * n + 1).to(BF)
    for plain in (None, b[:n]):
        with pytest.raises(Launched):
            call(x, w, plain)
    for other in (b[:1], b[:n].view(1, n), torch.randn(rows, n).to(BF), b[:1].expand(n), b[:2 * n:2]):
        _by_library(call, x, w, other)
    for refused in (torch.randn(n), b[:n - 1]):
        with pytest.raises(RuntimeError):
            call(x, w, refused)


@pytest.mark.parametrize("rows,k,kernel", [(8, 512, True), (9, 512, False), (16, 896, False), (16, 1024, True)])
def test_short_rows_of_narrow_projections(rows, k, kernel):
    """More than 8 rows of fewer than 1024 values: the library was measured to be faster."""
    torch.manual_seed(k)
    x, w = torch.randn(rows, k).to(BF), torch.randn(2048, k).to(BF)
    if kernel:
        with pytest.raises(Launched):
            _linear(x, w, None)
    else:
        _by_library(_linear, x, w, None)


@pytest.mark.parametrize("m,n,k,kind,kernel", [
    (384, 512, 2048, "swiglu", True), (384, 512, 2112, "swiglu", False), (321, 4160, 1024, "swiglu", True),
    (300, 1024, 8192, "norm", True), (1024, 1088, 1536, "norm", True), (1024, 1088, 1600, "norm", False),
    (300, 1024, 1536, "plain", True), (300, 1024, 1600, "plain", False), (300, 960, 1024, "plain", True),
    (300, 960, 1088, "plain", False), (300, 3072, 1536, "plain", True), (300, 3136, 1088, "plain", False),
    (300, 4160, 512, "plain", False), (300, 4224, 512, "plain", True), (300, 4160, 512, "norm", False)])
def test_lines_of_the_tiled_form(m, n, k, kind, kernel):
    """257 to 1024 rows: where the grid's idle CUs cost more than the library's split of K."""
    assert (hip.tiled_gemm_sizes(m, n, k, kind == "swiglu", kind == "norm") is not None) == kernel
