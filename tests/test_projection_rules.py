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
