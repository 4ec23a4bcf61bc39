"""Recurrences with a decay per key channel over prompt portions in chunks (``csrc/hybrid/hybrid_channel_chunks.hip``)
against the token-by-token form in fp64, and against the kernel that takes the recurrence literally (reached with value
rows that are no whole 16-byte runs): portions around a block of 16 and a chunk of 64 tokens, head sizes at the edges
of the instances, state carried in, sequences without rows or without a slot, rows of no sequence."""
import random

import pytest
import torch

from minivllm_amd.ops import hip_hybrid as hk

LENS = [1, 15, 0, 16, 17, 63, 64, 65, 129, 200, 5, 600]
PAST = [0, 9, 0, 0, 3, 0, 70, 0, 0, 1, 0, 2]
SLOTS = [3, 1, 2, 0, 12, 5, 7, 6, 8, 11, -1, 10]
HEAD, TAIL = 2, 3                                      # rows ahead of the first and behind the last sequence
TAU = 16.0


def layout():
    cu = [HEAD]
    for n in LENS:
        cu.append(cu[-1] + n)
    pos = [0] * HEAD + [p + i for n, p in zip(LENS, PAST) for i in range(n)] + [0] * TAIL
    return cu, pos


def make(rule, H, D, E, dtype, fast, seed):
    g = torch.Generator().manual_seed(seed)
    cu, pos = layout()
    T = cu[-1] + TAIL
    x = dict(q=torch.randn(T, H, D, generator=g), k=torch.randn(T, H, D, generator=g), v=torch.randn(T, H, E, generator=g),
             a=torch.randn(T, H * D, generator=g) * (12 if fast else 1))
    x = {n: t.to(dtype) for n, t in x.items()}
    # fast: decays of 1e-6 (GLA) and 0 (WKV) beside ones that hardly decay
    bias = torch.randn(H * D, generator=g) - (3 if rule == "wkv" else 0)
    return cu, pos, x, bias, torch.randn(H, D, generator=g) * 0.5, torch.randn(13, H, D, E, generator=g)


def call(rule, cu, pos, x, bias, bonus, state, pad, tau=TAU):
    """``pad``: numbers behind each value row."""
    T, H, E = x["v"].shape
    v = torch.zeros(T, H * E + pad, dtype=x["v"].dtype, device="cuda")
    v[:, :H * E] = x["v"].reshape(T, -1).cuda()
    v = v[:, :H * E].view(T, H, E)
    lay = [torch.tensor(t, dtype=torch.int32).cuda() for t in (cu, pos, SLOTS)]
    st = state.cuda()
    q, k, a = (x[n].cuda() for n in "qka")
    if rule == "gla":
        o = hk.gla_scan(q, k, v, a, bias.cuda(), tau, st, *lay, max(LENS))
    else:
        o = hk.wkv_scan(q, k, v, a, bias.cuda(), bonus.cuda(), st, *lay, max(LENS))
    return o.cpu(), st.cpu()


def decays(rule, a, bias, tau=TAU):
    z = a.double() + bias.double()
    return torch.exp(torch.nn.functional.logsigmoid(z) / tau) if rule == "gla" else torch.exp(-torch.exp(z))


def exact(rule, cu, x, bias, bonus, state, tau=TAU):
    T, H, D = x["q"].shape
    q, k, v = (x[n].double() for n in "qkv")
    if rule == "gla":
        q = q * D ** -0.5
    g = decays(rule, x["a"], bias, tau).view(T, H, D)
    o, want = torch.zeros(v.shape, dtype=torch.float64), state.double()
    for b, s in enumerate(SLOTS):
        if s < 0 or not LENS[b]:
            continue
        S = want[s] * (PAST[b] > 0)
        for t in range(cu[b], cu[b + 1]):
            kv = k[t][:, :, None] * v[t][:, None]
            N = g[t][:, :, None] * S + kv
            o[t] = torch.einsum("hde,hd->he", S + bonus.double()[:, :, None] * kv if rule == "wkv" else N, q[t])
            S = N
        want[s] = S
    return o, want


def off(got, want):
    return float((got.double().cpu() - want).norm() / want.norm().clamp_min(1e-30))


def owned(cu, T):
    m = torch.zeros(T, dtype=torch.bool)
    for b, s in enumerate(SLOTS):
        m[cu[b]:cu[b + 1]] = s >= 0
    return m


@pytest.mark.gpu
@pytest.mark.parametrize("rule,H,D,E", [("gla", 2, 64, 128), ("gla", 3, 48, 40), ("gla", 1, 4, 8), ("gla", 2, 36, 72),
                                        ("wkv", 2, 64, 64), ("wkv", 3, 48, 48), ("wkv", 1, 5, 16), ("wkv", 2, 64, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("fast", [False, True])
def test_scan(rule, H, D, E, dtype, fast):
    args = make(rule, H, D, E, dtype, fast, D + E)
    got, literal = (call(rule, *args, pad) for pad in ((-H * E) % 8, (-H * E) % 8 + 1))
    cu, _, x, bias, bonus, state = args
    want = exact(rule, cu, x, bias, bonus, state)
    for i, (y, z, w) in enumerate(zip(got, literal, want)):
        # the same sums in fp32, rounded in other places: twice the literal kernel's error and one rounding in the mean
        assert off(y, w) <= 2 * off(z, w) + 2.0 ** -26, (i, off(y, w), off(z, w))
    m = owned(cu, got[0].shape[0])
    assert not got[0][~m].any() and not literal[0][~m].any()


@pytest.mark.gpu
@pytest.mark.parametrize("rule,D,E", [("gla", 64, 128), ("wkv", 64, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_bits(rule, D, E, dtype):
    """Operands in parts lose nothing against the fp32 arithmetic of the literal kernel (a tenth for the sample's spread)."""
    args = make(rule, 4, D, E, dtype, False, 1)
    got, literal = (call(rule, *args, pad) for pad in (0, 1))
    cu, _, x, bias, bonus, state = args
    for y, z, w in zip(got, literal, exact(rule, cu, x, bias, bonus, state)):
        print(rule, dtype, off(y, w), off(z, w))
        assert off(y, w) <= 1.1 * off(z, w), (off(y, w), off(z, w))


@pytest.mark.gpu
@pytest.mark.parametrize("tau", [0.25, 1.0, 5.0, 16.0])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_slow_decays(tau, dtype):
    """A decay that stays what it is over a portion multiplies its error up: no more than the literal kernel's (and a tenth, for
    products in another order)."""
    cu, pos, x, _, bonus, state = make("gla", 2, 64, 64, dtype, False, 9)
    x["a"].zero_()
    bias = torch.linspace(3, 20, 128)
    args = (cu, pos, x, bias, bonus, state)
    got, literal = (call("gla", *args, pad, tau) for pad in (0, 1))
    for y, z, w in zip(got, literal, exact("gla", cu, x, bias, bonus, state, tau)):
        print(tau, dtype, off(y, w), off(z, w))
        assert off(y, w) <= 1.1 * off(z, w), (off(y, w), off(z, w))


@pytest.mark.gpu
@pytest.mark.parametrize("rule,D,E", [("gla", 64, 128), ("wkv", 48, 48)])
@pytest.mark.parametrize("name", ["q", "k", "v", "a"])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_not_finite(rule, D, E, name, bad):
    """What is not finite reaches no earlier token and no other sequence: the same places as token by token."""
    args = make(rule, 2, D, E, torch.bfloat16, False, 3)
    cu, x = args[0], args[2]
    x[name].view(x[name].shape[0], 2, -1)[cu[9] + 77, 1, 3] = bad
    got, literal = (call(rule, *args, pad) for pad in ((-2 * E) % 8, (-2 * E) % 8 + 1))
    for y, z in zip(got, literal):
        same = (y == z) | (y.isnan() & z.isnan()) | ((y - z).abs() <= 1e-4 * (1 + z.abs()))
        assert bool(same.all()), int((~same).sum())
    assert torch.isfinite(got[0][:cu[9] + 77]).all() and torch.isfinite(got[0][cu[10]:]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("H,D,E,wide", [(2, 64, 128, False), (3, 48, 40, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_normed(H, D, E, wide, dtype):
    cu, pos, x, bias, bonus, state = make("gla", H, D, E, dtype, False, 5)
    T = x["q"].shape[0]
    g = torch.Generator().manual_seed(6)
    gate = torch.randn(T, H * E, generator=g).to(dtype)
    w = (1 + 0.1 * torch.randn(H * E if wide else E, generator=g)).cuda()
    proj = torch.cat([x["q"].view(T, -1), x["k"].view(T, -1), x["v"].view(T, -1), gate], 1).cuda()
    gate, st, lay = gate.cuda(), state.cuda(), [torch.tensor(t, dtype=torch.int32).cuda() for t in (cu, pos, SLOTS)]
    y = hk.gla_norm(proj, x["a"].cuda(), (H, D, E), bias.cuda(), TAU, w, st, *lay, 1e-6, dtype, max(LENS)).view(T, H, E)
    o, st2 = call("gla", cu, pos, x, bias, bonus, state, 0)
    want = hk.gated_head_norm(o.cuda(), w, gate, 1e-6, dtype)
    assert torch.equal(st.cpu(), st2)
    step = 2.0 ** -7 if dtype == torch.bfloat16 else 1e-5            # sums in another order; then a rounding
    assert bool(((y - want).abs().float() <= step * want.abs().float() + 1e-6).all())
    assert not y[~owned(cu, T).cuda()].any()


@pytest.mark.parametrize("T,B,longest,H,D,E,norm,dt,chunks", [
    # 8 heads of 64 x 128, normed in the same call: a portion (30 us either way at 64 tokens), 64 of them
    (64, 1, 64, 8, 64, 128, 1, 0, False), (128, 1, 128, 8, 64, 128, 1, 0, True), (128, 1, 0, 8, 64, 128, 1, 0, True),
    (4096, 64, 64, 8, 64, 128, 1, 0, False), (8192, 64, 128, 8, 64, 128, 1, 0, True), (8192, 64, 128, 8, 64, 128, 1, 2, True),
    # many short portions; one long one among them
    (16384, 256, 64, 8, 32, 32, 1, 0, False), (16384, 256, 64, 8, 32, 32, 1, 2, False), (16384, 64, 256, 8, 32, 32, 1, 0, False),
    (2048, 8, 256, 8, 32, 32, 1, 0, True), (8192, 128, 64, 16, 64, 64, 1, 0, False), (2048, 32, 64, 16, 64, 64, 1, 0, False),
    (383, 256, 128, 8, 64, 128, 1, 0, False), (767, 256, 512, 8, 64, 128, 1, 0, True),
    # without the norm
    (96, 1, 96, 16, 64, 64, 0, 0, True), (95, 1, 95, 16, 64, 64, 0, 0, False), (768, 8, 96, 16, 64, 64, 0, 0, True),
    (4096, 32, 128, 16, 64, 64, 0, 0, False), (8192, 32, 256, 16, 64, 64, 0, 0, True)])
def test_lengths_that_pay(T, B, longest, H, D, E, norm, dt, chunks):
    assert bool(hk._chan_bytes(T, B, longest, H, D, E, 1, norm, dt)) == chunks
    assert hk._chan_bytes(T, B, -1, H, D, E, 1, norm, dt)                      # (what it would want)
    assert not hk._chan_bytes(T, B, longest, H, D, E, 0, norm, dt)            # addresses
    for D, E in ((72, 128), (64, 136), (64, 36), (2, 64)):                    # sizes without an instance
        assert not hk._chan_bytes(T, B, longest, H, D, E, 1, norm, dt)


@pytest.mark.parametrize("tokens,seqs", [(16384, 256), (4096, 512), (1100, 512), (64, 8), (9, 4), (1, 1), (2000, 2000)])
@pytest.mark.parametrize("D,E", [(64, 128), (48, 48), (128, 128)])
def test_no_step_takes_more(tokens, seqs, D, E):
    most = hk.channel_scan_workspace(tokens, seqs, 8, D, E)
    r, top = random.Random(tokens), 0
    steps = [(tokens, b) for b in range(1, min(seqs, tokens) + 1)]
    steps += [(t, r.randint(1, min(seqs, t))) for t in (r.randint(1, tokens) for _ in range(2000))]
    for t, b in steps:
        for longest in (0, t - b + 1):
            top = max(top, hk._chan_bytes(t, b, longest, 8, D, E, 1, 0, 0), hk._chan_bytes(t, b, longest, 8, D, E, 1, 1, 2))
    assert top <= most and (most <= 2 * top or tokens < 128)
