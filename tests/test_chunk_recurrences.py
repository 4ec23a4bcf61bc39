"""Recurrences over prompt portions in chunks on the matrix cores (``csrc/hybrid/hybrid_chunks.hip``)
against the token-by-token form in fp64, and against the kernel that takes the recurrence literally
(reached with the same numbers in rows that are no whole 16-byte runs): portions around a block of 16
and a chunk of 64 tokens, head sizes at the edges of the instances, state carried in, sequences
without rows or without a slot, rows of no sequence."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from minivllm_amd.ops import hip_hybrid as hk

LENS = [1, 15, 0, 16, 17, 63, 64, 65, 129, 200, 5]
PAST = [0, 9, 0, 0, 3, 0, 70, 0, 0, 1, 0]
SLOTS = [3, 1, 2, 0, 12, 5, 7, 6, 8, 11, -1]
TAIL = 3                                               # rows behind the last sequence


def layout():
    cu = [0]
    for n in LENS:
        cu.append(cu[-1] + n)
    pos = [p + i for n, p in zip(LENS, PAST) for i in range(n)] + [0] * TAIL
    return cu, [torch.tensor(x, dtype=torch.int32).cuda() for x in (cu, pos, SLOTS)]


def off(got, want):
    return float((got.double().cpu() - want).norm() / want.norm().clamp_min(1e-30))


@pytest.mark.parametrize("H,D,E", [(2, 128, 128), (1, 8, 8), (3, 48, 40), (2, 64, 72), (1, 72, 32), (2, 120, 64)])
@pytest.mark.parametrize("cap", [4.0, 15.0])
def test_mlstm(H, D, E, cap):
    g = torch.Generator().manual_seed(D + E)
    cu, lay = layout()
    T, Z, NS = cu[-1] + TAIL, (E + 15) // 16, 13
    n_in = 2 * H * D + H * E + 2 * H
    proj = torch.randn(T, n_in, generator=g)
    proj[:, 2 * H * D + H * E:] *= 4                   # gates that reach the cap
    proj = proj.bfloat16()
    bi, bf = torch.randn(H, generator=g), 2 + torch.randn(H, generator=g)
    init = [torch.randn(NS, H, D, E, generator=g), torch.randn(NS, H, 1, D, generator=g).expand(-1, -1, Z, -1).contiguous(),
            torch.randn(NS, H, 1, generator=g).expand(-1, -1, Z).contiguous()]

    def run(pad):
        p = torch.zeros(T, n_in + pad, dtype=torch.bfloat16).cuda()
        p[:, :n_in] = proj.cuda()
        q, k, v, i, f = p[:, :n_in].split([H * D, H * D, H * E, H, H], -1)
        st = [x.cuda() for x in init]
        o = hk.mlstm_scan(q.view(T, H, D), k.view(T, H, D), v.view(T, H, E), i, f, bi.cuda(), bf.cuda(), cap, *st, *lay)
        return [o.cpu()] + [x.cpu() for x in st]

    q, k, v, i, f = proj.double().split([H * D, H * D, H * E, H, H], -1)
    q, k, v = q.view(T, H, D) * D ** -0.5, k.view(T, H, D), v.view(T, H, E)
    i = cap * torch.tanh((i + bi.double()) / cap)
    f = torch.nn.functional.logsigmoid(cap * torch.tanh((f + bf.double()) / cap))
    o = torch.zeros(T, H, E, dtype=torch.float64)
    want = [x.double() for x in init]
    for b, (n, s) in enumerate(zip(LENS, SLOTS)):
        if s < 0 or n == 0:
            continue
        S, N, m = (x[s].clone() * (PAST[b] > 0) for x in want)
        N, m = N[:, 0], m[:, 0]
        for t in range(cu[b], cu[b + 1]):
            m2 = torch.maximum(f[t] + m, i[t])
            a, c = torch.exp(f[t] + m - m2), torch.exp(i[t] - m2)
            S = a[:, None, None] * S + c[:, None, None] * k[t][:, :, None] * v[t][:, None]
            N = a[:, None] * N + c[:, None] * k[t]
            m = m2
            den = torch.maximum((N * q[t]).sum(-1).abs(), torch.exp(-m)) + 1e-6
            o[t] = torch.einsum("hde,hd->he", S, q[t]) / den[:, None]
        want[0][s], want[1][s], want[2][s] = S, N[:, None], m[:, None]
    got, literal = run((-n_in) % 8), run((-n_in) % 8 + 1)
    for x, y, w in zip(got, literal, [o] + want):
        # the same sums in fp32, rounded in other places: twice the literal kernel's error and one rounding in the
        # mean (a part of eight bits less in any operand is 2^-17)
        assert off(x, w) <= 2 * off(y, w) + 2.0 ** -26, (off(x, w), off(y, w))
    owned = torch.zeros(T, dtype=torch.bool)
    for b, s in enumerate(SLOTS):
        owned[cu[b]:cu[b + 1]] = s >= 0
    for x in (got[0], literal[0]):
        assert bool((x[~owned] == 0).all())


@pytest.mark.parametrize("H,G,D,E", [(2, 1, 128, 128), (3, 3, 8, 4), (4, 2, 48, 40), (2, 2, 64, 72), (6, 2, 72, 32), (33, 11, 120, 64)])
@pytest.mark.parametrize("correct", [True, False])
@pytest.mark.parametrize("fast", [True, False])
def test_delta_rule(H, G, D, E, correct, fast):
    """``fast``: decays down to 1e-9 per token (their products leave fp32's range inside a chunk), keys that
    repeat each other."""
    g = torch.Generator().manual_seed(D + E)
    cu, lay = layout()
    T, NS = cu[-1] + TAIL, 13
    q, k = (torch.randn(T, G, D, generator=g) for _ in range(2))
    if fast:
        k = k[torch.arange(T) // 3]
    q, k = q / q.norm(dim=-1, keepdim=True) * D ** -0.5, k / k.norm(dim=-1, keepdim=True)
    v, beta = torch.randn(T, H, E, generator=g), torch.sigmoid(2 * torch.randn(T, H, generator=g))
    decay = torch.exp(-torch.rand(T, H, generator=g) * (20.0 if fast else 0.2))
    if fast:
        decay[::7] = 1.0
    state = torch.randn(NS, H, D, E, generator=g)

    def run(shift):                                    # rows that do not start on 16 bytes go token by token
        st = state.cuda()
        return hk.delta_scan(at(q, shift), at(k, shift), at(v, shift), beta.cuda(), decay.cuda(), st, *lay, correct).cpu(), st.cpu()

    qd, kd = (x.double().repeat_interleave(H // G, 1) for x in (q, k))
    o, want = torch.zeros(T, H, E, dtype=torch.float64), state.double()
    for b, (n, s) in enumerate(zip(LENS, SLOTS)):
        if s < 0:
            continue
        S = want[s] * (PAST[b] > 0)
        for t in range(cu[b], cu[b + 1]):
            S = S * decay[t].double()[:, None, None]
            u = beta[t].double()[:, None] * (v[t].double() - (torch.einsum("hde,hd->he", S, kd[t]) if correct else 0))
            S = S + kd[t][:, :, None] * u[:, None]
            o[t] = torch.einsum("hde,hd->he", S, qd[t])
        want[s] = S
    got, literal = run(0), run(1)
    for x, y, w in zip(got, literal, (o, want)):
        assert off(x, w) <= 2 * off(y, w) + 2.0 ** -26, (off(x, w), off(y, w))      # as above
    owned = torch.zeros(T, dtype=torch.bool)
    for b, s in enumerate(SLOTS):
        owned[cu[b]:cu[b + 1]] = s >= 0
    for x in (got[0], literal[0]):
        assert bool((x[~owned] == 0).all())


def at(x, shift):
    """x on the GPU, ``shift`` numbers behind a 16-byte address."""
    y = torch.empty(x.numel() + shift, dtype=x.dtype, device="cuda")
    y[shift:] = x.reshape(-1).cuda()
    return y[shift:].view(x.shape)


def portions(B, n):
    return [torch.tensor(x, dtype=torch.int32).cuda() for x in (list(range(0, B * n + 1, n)), list(range(n)) * B, list(range(B)))]


@pytest.mark.parametrize("n", [200, 512])
@pytest.mark.parametrize("correct", [True, False])
def test_bits_of_the_delta_rule(n, correct):
    """Operands in parts lose nothing against the fp32 arithmetic of the literal kernel: over decays of a trained
    range neither the outputs nor the state are further from 64 bits (a tenth for the sample's own spread)."""
    g = torch.Generator().manual_seed(n)
    B, H, G, D, E = 2, 4, 2, 128, 128
    T = B * n
    q, k = (torch.nn.functional.normalize(torch.randn(T, G, D, generator=g), dim=-1) for _ in range(2))
    q, v, beta = q * D ** -0.5, torch.randn(T, H, E, generator=g), torch.sigmoid(torch.randn(T, H, generator=g))
    rate = 1 + 15 * torch.rand(H, generator=g)
    decay = torch.exp(-rate * torch.nn.functional.softplus(torch.randn(T, H, generator=g) - 4.6))
    lay = portions(B, n)
    args = [x.cuda() for x in (beta, decay)]
    got = []
    for shift in (0, 1):
        st = torch.zeros(B, H, D, E, device="cuda")
        got.append((hk.delta_scan(at(q, shift), at(k, shift), at(v, shift), *args, st, *lay, correct), st))
    qd, kd = (x.cuda().double().repeat_interleave(H // G, 1).view(B, n, H, D) for x in (q, k))
    vd, bd, gd = v.cuda().double().view(B, n, H, E), args[0].double().view(B, n, H), args[1].double().view(B, n, H)
    S, o = torch.zeros(B, H, D, E, dtype=torch.float64, device="cuda"), torch.empty(B, n, H, E, dtype=torch.float64, device="cuda")
    for t in range(n):
        S = S * gd[:, t, :, None, None]
        u = vd[:, t] - (torch.matmul(kd[:, t, :, None], S)[:, :, 0] if correct else 0)
        S = S + kd[:, t, :, :, None] * (bd[:, t, :, None] * u)[:, :, None]
        o[:, t] = torch.matmul(qd[:, t, :, None], S)[:, :, 0]
    for x, y, w in zip(*got, (o.view(T, H, E), S)):
        chunks, literal = off(x, w.cpu()), off(y, w.cpu())
        assert chunks <= 1.1 * literal, (chunks, literal)


@pytest.mark.parametrize("forget", [4.0, 0.0])
def test_bits_of_the_matrix_lstm(forget):
    """As above; a row's error is counted against the row, as small denominators make some rows a thousand times the
    others, and the running maximum's against its last bit.  (W_end v is rounded once more than in the literal kernel:
    2^-26 in the mean, which shows where little else is rounded, as with half of the state forgotten per token.)"""
    g = torch.Generator().manual_seed(int(forget))
    B, n, H, D, E, cap = 2, 500, 4, 128, 128, 15.0
    T, n_in = B * n, 2 * H * D + H * E + 2 * H
    proj = torch.randn(T, n_in, generator=g)
    proj[:, -2 * H:] *= 2
    proj = proj.bfloat16().cuda()
    bi, bf = torch.randn(H, generator=g).cuda(), (forget + torch.randn(H, generator=g)).cuda()
    lay, got = portions(B, n), []
    for pad in ((-n_in) % 8, (-n_in) % 8 + 1):
        p = torch.zeros(T, n_in + pad, dtype=torch.bfloat16, device="cuda")
        p[:, :n_in] = proj
        q, k, v, i, f = p[:, :n_in].split([H * D, H * D, H * E, H, H], -1)
        st = [torch.zeros(B, H, D, E, device="cuda"), torch.zeros(B, H, E // 16, D, device="cuda"),
              torch.zeros(B, H, E // 16, device="cuda")]
        got.append([hk.mlstm_scan(q.view(T, H, D), k.view(T, H, D), v.view(T, H, E), i, f, bi, bf, cap, *st, *lay)] + st)
    q, k, v, i, f = proj.double().split([H * D, H * D, H * E, H, H], -1)
    q, k, v = q.view(B, n, H, D) * D ** -0.5, k.view(B, n, H, D), v.view(B, n, H, E)
    i = (cap * torch.tanh((i + bi.double()) / cap)).view(B, n, H)
    f = torch.nn.functional.logsigmoid(cap * torch.tanh((f + bf.double()) / cap)).view(B, n, H)
    S, o = torch.zeros(B, H, D, E, dtype=torch.float64, device="cuda"), torch.empty(B, n, H, E, dtype=torch.float64, device="cuda")
    N, m = S[..., 0].clone(), S[..., 0, 0].clone()
    for t in range(n):
        m2 = torch.maximum(f[:, t] + m, i[:, t])
        a, c = torch.exp(f[:, t] + m - m2), torch.exp(i[:, t] - m2)
        S = a[..., None, None] * S + c[..., None, None] * k[:, t, :, :, None] * v[:, t, :, None]
        N, m = a[..., None] * N + c[..., None] * k[:, t], m2
        den = torch.maximum((N * q[:, t]).sum(-1).abs(), torch.exp(-m)) + 1e-6
        o[:, t] = torch.matmul(q[:, t, :, None], S)[:, :, 0] / den[..., None]
    rows = [float(((x[0].double() - o.view(T, H, E)).norm(dim=-1) / o.view(T, H, E).norm(dim=-1)).median()) for x in got]
    assert rows[0] <= 1.1 * rows[1], rows
    for x, y, w in zip(got[0][1:3], got[1][1:3], (S, N[:, :, None].expand(-1, -1, E // 16, -1))):
        chunks, literal = off(x, w.cpu()), off(y, w.cpu())
        assert chunks <= 1.1 * literal + 2.0 ** -26, (chunks, literal)
    assert off(got[0][3], m[..., None].expand(-1, -1, E // 16).cpu()) <= 2.0 ** -23


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,D,E,taps", [(2, 1, 8, 8, 4), (1, 1, 48, 40, 2), (3, 1, 16, 24, 3), (2, 2, 128, 64, 4),
                                          # heads that are no whole runs in rows that are, rows that are none
                                          (4, 2, 12, 16, 4), (2, 2, 20, 4, 2), (8, 4, 6, 3, 3), (3, 1, 10, 7, 4), (2, 1, 8, 8, 6)])
@pytest.mark.parametrize("ssd,channel", [(False, False), (False, True), (True, False)])
def test_delta_prepare_rows(dt, H, G, D, E, taps, ssd, channel):
    """Several rows per workgroup: portions that start, end or lie inside its rows, shorter than the taps, with
    and without a past, without a slot; then a step of single tokens on the tails it left."""
    from minivllm_amd.ops import torch_seqmix as ref
    g = torch.Generator().manual_seed(taps)
    lens = [1, 2, 3, 700, 1, 0, 1500, 7, 9, 16, 2000, 5, 1, 2]
    past = [5, 0, 9, 3, 0, 0, 0, 4, 0, 2, 8, 0, 3, 7]
    slots = torch.tensor([3, 0, 12, 7, 13, 2, 1, 9, -1, 10, 11, 4, 5, 6], dtype=torch.int32)
    cu = torch.tensor([0] + lens).cumsum(0).int()
    T, C, N = int(cu[-1]), 2 * G * D + H * E, (H * D if channel else H)
    pos = torch.cat([torch.arange(p, p + n) for n, p in zip(lens, past)]).int()
    row_seq = torch.cat([torch.full((n,), b) for b, n in enumerate(lens)]).int()
    conv_w, conv_b = torch.randn(C, taps, generator=g), torch.randn(C, generator=g) if ssd else None
    a_log, dt_bias = torch.randn(H, generator=g), torch.randn(N, generator=g)
    tail = torch.randn(14, taps - 1, C, generator=g)
    width = -(-(C + H + N) // 8) * 8
    steps = [(torch.randn(T, width, generator=g).to(dt), cu, pos, row_seq),
             (torch.randn(14, width, generator=g).to(dt), None, torch.tensor([p + n for n, p in zip(lens, past)]).int(), None)]

    def run(f, to):
        st, outs = to(tail.clone()), []
        for proj, c, p, rs in steps:
            x = to(proj)
            q, k, v, b, a = x[:, :C + H + N].split([G * D, G * D, H * E, H, N], -1)
            n = x.shape[0]
            args = [q.view(n, G, D), k.view(n, G, D), v.view(n, H, E), b, a, to(conv_w), to(a_log), to(dt_bias), st,
                    None if c is None else to(c), to(p), to(slots)]
            kw = dict(conv_bias=None if conv_b is None else to(conv_b), ssd=ssd)
            if f is hk.delta_prepare:
                kw["row_seq"] = None if rs is None else to(rs)
            outs.append([y.cpu() for y in f(*args, **kw)])
        return outs, st.cpu()

    (w1, w2), wt = run(ref.delta_prepare, lambda x: x)
    (g1, g2), gt = run(hk.delta_prepare, lambda x: x.cuda())
    live = [(slots[row_seq.long()] >= 0), slots >= 0]
    for got, want, ok in ((g1, w1, live[0]), (g2, w2, live[1])):
        for x, y in zip(got, want):
            # silu, softplus, exp and sums of up to 128 squares in fp32
            torch.testing.assert_close(x[ok], y[ok], rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(gt, wt, rtol=0, atol=0)


@pytest.mark.parametrize("H,G,D,E", [(4, 2, 128, 128), (2, 2, 8, 16), (3, 1, 100, 32), (2, 1, 256, 64), (1, 1, 33, 256), (2, 1, 64, 64)])
@pytest.mark.parametrize("rule", ["delta", "channel", "plain"])
def test_single_tokens(H, G, D, E, rule):
    g = torch.Generator().manual_seed(D * E)
    B = 7
    slots = torch.tensor([2, 0, -1, 5, 4, 1, 3], dtype=torch.int32)
    pos = torch.tensor([3, 0, 4, 9, 1, 0, 2], dtype=torch.int32)
    q, k = (torch.randn(B, G, D, generator=g) for _ in range(2))
    k = k / k.norm(dim=-1, keepdim=True)
    v, beta = torch.randn(B, H, E, generator=g), torch.rand(B, H, generator=g)
    decay = torch.rand(B, H, D, generator=g) if rule == "channel" else torch.rand(B, H, generator=g)
    state = torch.randn(6, H, D, E, generator=g)
    gs = state.cuda()
    got = hk.delta_scan(q.cuda(), k.cuda(), v.cuda(), beta.cuda(), decay.cuda(), gs, None, pos.cuda(), slots.cuda(),
                        rule != "plain").cpu()
    qd, kd = (x.double().repeat_interleave(H // G, 1) for x in (q, k))
    want, ws = torch.zeros(B, H, E, dtype=torch.float64), state.double()
    for b, s in enumerate(slots.tolist()):
        if s < 0:
            continue
        d = decay[b].double()
        S = ws[s] * (int(pos[b]) > 0) * (d[:, :, None] if rule == "channel" else d[:, None, None])
        u = beta[b].double()[:, None] * (v[b].double() - (torch.einsum("hde,hd->he", S, kd[b]) if rule != "plain" else 0))
        ws[s] = S + kd[b][:, :, None] * u[:, None]
        want[b] = torch.einsum("hde,hd->he", ws[s], qd[b])
    # sums of up to 256 fp32 products
    assert off(got, want) <= 256 * 2.0 ** -24 and off(gs, ws) <= 256 * 2.0 ** -24
    assert bool((got[2] == 0).all())


@pytest.mark.parametrize("H,G,D,E", [(16, 8, 128, 128), (8, 4, 64, 64), (4, 4, 256, 64), (2, 2, 64, 256), (8, 8, 128, 16)])
@pytest.mark.parametrize("rule", ["delta", "channel", "plain"])
def test_bits_of_single_tokens(H, G, D, E, rule):
    """Neither the outputs nor the state are further from 64 bits than those of the token-by-token kernels, which
    take the same rows as portions of one token (a twentieth for the sample's spread)."""
    g = torch.Generator().manual_seed(D + E)
    B = 64
    q, k = (torch.nn.functional.normalize(torch.randn(B, G, D, generator=g), dim=-1).cuda() for _ in range(2))
    q = q * D ** -0.5
    v, beta = torch.randn(B, H, E, generator=g).cuda(), torch.rand(B, H, generator=g).cuda()
    decay = (0.7 + 0.3 * (torch.rand(B, H, D, generator=g) if rule == "channel" else torch.rand(B, H, generator=g))).cuda()
    state = torch.randn(B, H, D, E, generator=g).cuda()
    pos, slots = torch.ones(B, dtype=torch.int32).cuda(), torch.arange(B, dtype=torch.int32).cuda()
    got = []
    for cu in (None, torch.arange(B + 1, dtype=torch.int32).cuda()):
        st = state.clone()
        got.append((hk.delta_scan(q, k, v, beta, decay, st, cu, pos, slots, rule != "plain"), st))
    qd, kd = (x.double().repeat_interleave(H // G, 1) for x in (q, k))
    S = state.double() * (decay.double()[..., None] if rule == "channel" else decay.double()[..., None, None])
    u = v.double() - ((S * kd[..., None]).sum(2) if rule != "plain" else 0)
    S = S + kd[..., None] * (beta.double()[..., None] * u)[:, :, None]
    for x, y, w in zip(*got, ((S * qd[..., None]).sum(2), S)):
        single, literal = off(x, w.cpu()), off(y, w.cpu())
        assert single <= 1.05 * literal, (single, literal)


INF, NAN = float("inf"), float("nan")


def same_but_for_rounding(got, want):
    """Infinities and NaN in the same places, and elsewhere the same numbers (how closely is tested above: two
    roundings of a small denominator, 2^-23 of its terms, may differ by a thousand times that)."""
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[got.isinf()], want[want.isinf()])
    ok = want.isfinite()
    assert off(got[ok], want[ok].double()) <= 2.0 ** -13


@pytest.mark.parametrize("D,E", [(128, 128), (64, 72), (8, 8)])
@pytest.mark.parametrize("what", ["k inf", "k nan", "v inf", "v nan", "q inf", "f nan", "i nan", "state inf"])
def test_mlstm_infinities(D, E, what):
    """What is not finite reaches the outputs and states that it reaches token by token, and no earlier token, no
    other column, no other sequence."""
    g = torch.Generator().manual_seed(D)
    H, cap = 2, 15.0
    cu, lay = layout()
    T, Z, NS = cu[-1] + TAIL, (E + 15) // 16, 13
    n_in = 2 * H * D + H * E + 2 * H
    proj = torch.randn(T, n_in, generator=g)
    bi, bf = torch.randn(H, generator=g), 4 + torch.randn(H, generator=g)
    init = [torch.randn(NS, H, D, E, generator=g), torch.randn(NS, H, 1, D, generator=g).expand(-1, -1, Z, -1).contiguous(),
            torch.randn(NS, H, 1, generator=g).expand(-1, -1, Z).contiguous()]
    t, h = cu[8] + 70, 1                               # token 70 of 129: its chunk has tokens ahead of it
    x = INF if "inf" in what else NAN
    at = {"k": H * D + h * D + 3, "v": 2 * H * D + h * E + E // 2, "q": h * D + 5, "i": n_in - 2 * H + h, "f": n_in - H + h}
    if what[0] in at:
        proj[t, at[what[0]]] = x
    else:
        init[0][SLOTS[6], h, 2, 1] = x                 # (a sequence with a past)
    proj = proj.bfloat16()

    def run(pad):
        p = torch.zeros(T, n_in + pad, dtype=torch.bfloat16).cuda()
        p[:, :n_in] = proj.cuda()
        q, k, v, i, f = p[:, :n_in].split([H * D, H * D, H * E, H, H], -1)
        st = [y.cuda() for y in init]
        o = hk.mlstm_scan(q.view(T, H, D), k.view(T, H, D), v.view(T, H, E), i, f, bi.cuda(), bf.cuda(), cap, *st, *lay)
        return [o.cpu()] + [y.cpu() for y in st]

    got, literal = run((-n_in) % 8), run((-n_in) % 8 + 1)
    assert not bool(got[0].isfinite().all()) and bool(got[0][cu[8]:t].isfinite().all())
    for y, w in zip(got, literal):
        same_but_for_rounding(y, w)


@pytest.mark.parametrize("H,G,D,E", [(2, 1, 128, 128), (40, 40, 64, 72), (2, 1, 8, 4)])
@pytest.mark.parametrize("correct", [True, False])
@pytest.mark.parametrize("what", ["k inf", "k nan", "v inf", "v nan", "q inf", "beta nan", "decay nan", "state inf", "large"])
def test_delta_infinities(H, G, D, E, correct, what):
    """As above; ``large``: a finite value whose rounded part is none.  (40 heads of 72 columns: 64 per workgroup.)"""
    g = torch.Generator().manual_seed(D)
    cu, lay = layout()
    T, NS, h = cu[-1] + TAIL, 13, H - 1
    q, k = (torch.nn.functional.normalize(torch.randn(T, G, D, generator=g), dim=-1) for _ in range(2))
    ops = {"q": q * D ** -0.5, "k": k, "v": torch.randn(T, H, E, generator=g), "beta": torch.rand(T, H, generator=g),
           "decay": torch.exp(-torch.rand(T, H, generator=g) * 0.2)}
    state = torch.randn(NS, H, D, E, generator=g)
    t, x, name = cu[8] + 70, INF if "inf" in what else NAN, what.split()[0]
    if name in ("q", "k"):
        ops[name][t, G - 1, 3] = x
    elif name in ("beta", "decay"):
        ops[name][t, h] = x
    elif name == "v":
        ops[name][t, h, E // 2] = x
    elif name == "large":
        ops["v"][t, h, E // 2], ops["beta"][t, h] = torch.finfo(torch.float32).max, 1.0
    else:
        state[SLOTS[6], h, 2, 1] = x

    def run(shift):
        st = state.cuda()
        o = hk.delta_scan(at(ops["q"], shift), at(ops["k"], shift), at(ops["v"], shift), ops["beta"].cuda(),
                          ops["decay"].cuda(), st, *lay, correct)
        return o.cpu(), st.cpu()

    got, literal = run(0), run(1)
    assert name == "large" or not bool(got[0].isfinite().all())
    assert bool(got[0][cu[8]:t].isfinite().all())
    for y, w in zip(got, literal):
        same_but_for_rounding(y / 2.0 ** 70, w / 2.0 ** 70) if name == "large" else same_but_for_rounding(y, w)
