"""The matrix LSTM's prompt portions in chunks, in both types, and its layer's call with the norm inside: portions around a chunk
and a block of 16, value columns around the kernels' blocks, pasts, rows of no sequence, infinities; against float64 and
against the recurrence token by token (an address off 16 bytes)."""
import pytest
import torch

from minivllm_amd.layers.linear_attention import MatrixLSTM

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from minivllm_amd.ops import hip_hybrid as hk

LENS, SLOTS, PAST, HEAD, TAIL = [64, 1, 200, 15, 63, 65, 130, 17, 16], [3, 0, 6, -1, 1, 5, 7, 2, 4], [0, 5, 3, 0, 0, 7, 0, 2, 0], 3, 4


def _layout():
    cu = [HEAD]
    for n in LENS:
        cu.append(cu[-1] + n)
    T = cu[-1] + TAIL
    pos = torch.zeros(T, dtype=torch.int32)
    for b, n in enumerate(LENS):
        pos[cu[b]:cu[b + 1]] = torch.arange(n) + PAST[b]
    i32 = lambda x: torch.as_tensor(x, dtype=torch.int32).cuda()
    return T, cu, (i32(cu), i32(pos), i32(SLOTS))


def _rows(proj, pad, lead):
    T, n = proj.shape
    p = torch.zeros(T * (n + pad) + lead, dtype=proj.dtype, device="cuda")[lead:].view(T, n + pad)
    p[:, :n] = proj.cuda()
    return p[:, :n]


def _exact(proj, H, D, E, bi, bf, cap, init, cu):
    """In float64: outputs and states, and the size of what is summed up in each: their errors are that many roundings, however
    much of it cancels (a row's denominator is |n . q|, whose terms can)."""
    q, k, v, _, i, f = proj.double().cuda().split([H * D, H * D, H * E, H * E, H, H], -1)
    T = proj.shape[0]
    q, k, v = q.view(T, H, D) * D ** -0.5, k.view(T, H, D), v.view(T, H, E)
    i = cap * torch.tanh((i + bi.double()) / cap)
    f = torch.nn.functional.logsigmoid(cap * torch.tanh((f + bf.double()) / cap))
    o = torch.zeros(T, H, E, dtype=torch.float64, device="cuda")
    st = [x.double() for x in init]
    size = [torch.zeros_like(o)] + [x.abs() for x in st]
    for b, slot in enumerate(SLOTS):
        if slot < 0:
            continue
        S, N, m = (st[0][slot].clone(), st[1][slot, :, 0].clone(), st[2][slot, :, 0].clone()) if PAST[b] else \
            (torch.zeros_like(st[0][slot]), torch.zeros_like(st[1][slot, :, 0]), torch.zeros_like(st[2][slot, :, 0]))
        Sa, Na, ma = S.abs(), N.abs(), m.abs()
        for t in range(cu[b], cu[b + 1]):
            m2 = torch.maximum(f[t] + m, i[t])
            fa, ia = torch.exp(f[t] + m - m2), torch.exp(i[t] - m2)
            S = fa[:, None, None] * S + ia[:, None, None] * k[t][:, :, None] * v[t][:, None]
            N = fa[:, None] * N + ia[:, None] * k[t]
            Sa = fa[:, None, None] * Sa + ia[:, None, None] * k[t].abs()[:, :, None] * v[t].abs()[:, None]
            Na = fa[:, None] * Na + ia[:, None] * k[t].abs()
            m, ma = m2, torch.maximum(ma + f[t].abs(), i[t].abs())
            den = torch.maximum((N * q[t]).sum(-1).abs(), torch.exp(-m)) + 1e-6
            o[t] = torch.matmul(q[t][:, None], S)[:, 0] / den[:, None]
            size[0][t] = (torch.matmul(q[t].abs()[:, None], Sa)[:, 0] + o[t].abs() * (Na * q[t].abs()).sum(-1)[:, None]) / den[:, None]
        st[0][slot], st[1][slot], st[2][slot] = S, N[:, None], m[:, None]
        size[1][slot], size[2][slot], size[3][slot] = Sa, Na[:, None], ma[:, None]
    return [o] + st, size


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,D,E", [(2, 128, 128), (3, 48, 40), (1, 64, 136), (2, 72, 264), (1, 8, 8),
                                   # more walks of 32 columns than CUs: bfloat16 in one kernel
                                   (15, 48, 40), (8, 64, 136), (29, 8, 8), (16, 64, 64)])
@pytest.mark.parametrize("gates", [1.0, 6.0])
def test_against_exact_and_tokens(dt, H, D, E, gates):
    g = torch.Generator().manual_seed(D + E)
    T, cu, lay = _layout()
    n, Z, cap = 2 * H * D + 2 * H * E + 2 * H, (E + 15) // 16, 15.0
    proj = torch.randn(T, n, generator=g)
    proj[:, -2 * H:] *= gates
    proj = proj.to(dt)
    bi, bf = torch.randn(H, generator=g).cuda(), (2 + torch.randn(H, generator=g)).cuda()
    init = [torch.randn(8, H, D, E, generator=g).cuda(), torch.randn(8, H, 1, D, generator=g).expand(-1, -1, Z, -1).contiguous().cuda(),
            torch.randn(8, H, 1, generator=g).expand(-1, -1, Z).contiguous().cuda()]

    def run(p):
        q, k, v, _, i, f = p.split([H * D, H * D, H * E, H * E, H, H], -1)
        st = [x.clone() for x in init]
        return [hk.mlstm_scan(q.view(T, H, D), k.view(T, H, D), v.view(T, H, E), i, f, bi, bf, cap, *st, *lay)] + st

    whole = -n % 8
    chunks, tokens = run(_rows(proj, whole, 0)), run(_rows(proj, whole, 1))
    owned = torch.zeros(T, dtype=torch.bool, device="cuda")
    for b, slot in enumerate(SLOTS):
        owned[cu[b]:cu[b + 1]] = slot >= 0
    assert not chunks[0][~owned].any()
    # Every value of every row, in roundings of what is summed up in it: a weight is a product of up to 64 rounded decays, and
    # sums of 64 and 128 terms come behind it.  (The recurrence, of 205 steps, comes to 40, the chunks to 33.)
    want, size = _exact(proj, H, D, E, bi, bf, cap, init, cu)
    off = lambda x, i: ((x.double() - want[i]).abs() / (size[i] + 1e-30)).flatten(1).amax(1) / 2.0 ** -24
    for i, (got, lit) in enumerate(zip(chunks, tokens)):
        a, b = off(got, i), off(lit, i)
        assert bool((a <= 64).all()) and bool((b <= 64).all()), (i, a, b)
        a, b = (float((x.double() - want[i]).abs().div(size[i] + 1e-30).pow(2).mean().sqrt()) for x in (got, lit))
        assert a <= 1.5 * b + 2.0 ** -26, (i, a, b)                 # and in the mean no more than token by token
    # infinities and NaNs: what the recurrence makes of them
    bad = proj.clone()
    bad[cu[2] + 70, 0] = float("inf")
    bad[cu[6] + 3, 2 * H * D + 1] = float("nan")
    bad[cu[7] + 1, -1] = float("nan")
    chunks, tokens = run(_rows(bad, whole, 0)), run(_rows(bad, whole, 1))
    for x, y in zip(chunks, tokens):
        assert torch.equal(x.isnan(), y.isnan()) and torch.equal(x.isinf(), y.isinf())
    # what stays finite met none of them, and is what it was without them
    for i, x in enumerate(chunks):
        fine = x.isfinite().flatten(2).all(-1) if i else x.isfinite().all(-1)
        assert bool(((x.double() - want[i]).abs() <= 64 * 2.0 ** -24 * size[i] + 1e-30)[fine].all()), i


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,D,E", [(2, 128, 128), (3, 48, 40), (3, 20, 24), (1, 64, 136), (15, 48, 40)])
@pytest.mark.parametrize("step", ["prompts", "tokens", "one"])
@pytest.mark.parametrize("extra", [0, 1])
def test_rows_call_is_the_two_calls(dt, H, D, E, step, extra):
    g = torch.Generator().manual_seed(D + E)
    if step == "prompts":
        T, cu, lay = _layout()
    else:
        T = 1 if step == "one" else 9
        lay = (None, torch.full((T,), 5, dtype=torch.int32, device="cuda"),
               torch.tensor([3, 0, -1, 1, 2, 4, 5, 6, 7][:T], dtype=torch.int32, device="cuda"))
    layer, Z = MatrixLSTM(H, D, E, 15.0, 1e-6).cuda(), (E + 15) // 16
    layer.norm_weight.data.normal_()
    proj = _rows(torch.randn(T, sum(layer.split_sizes()), generator=g).to(dt), extra, 0)
    init = [torch.randn(8, H, D, E, generator=g).cuda(), torch.randn(8, H, 1, D, generator=g).expand(-1, -1, Z, -1).contiguous().cuda(),
            torch.randn(8, H, 1, generator=g).expand(-1, -1, Z).contiguous().cuda()]
    one, two = [x.clone() for x in init], [x.clone() for x in init]
    y = hk.mlstm_norm(proj, (H, D, E), layer.i_bias, layer.f_bias, 15.0, layer.norm_weight, *one, *lay, 1e-6, dt)
    q, k, v, gate, i, f = proj.split(layer.split_sizes(), -1)
    o = hk.mlstm_scan(q.view(T, H, D), k.view(T, H, D), v.view(T, H, E), i, f, layer.i_bias, layer.f_bias, 15.0, *two, *lay)
    want = hk.gated_head_norm(o, layer.norm_weight, gate, 1e-6, dt, "sigmoid").view(T, H * E)
    assert torch.equal(y, want) and all(torch.equal(a, b) for a, b in zip(one, two))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,D,E", [(2, 64, 128), (3, 20, 24), (2, 128, 136)])
@pytest.mark.parametrize("T", [1, 9])
def test_gla_rows_call_is_the_two_calls(dt, H, D, E, T):
    g = torch.Generator().manual_seed(D + E)
    lay = (None, torch.full((T,), 5, dtype=torch.int32, device="cuda"),
           torch.tensor([3, 0, -1, 1, 2, 4, 5, 6, 7][:T], dtype=torch.int32, device="cuda"))
    proj = torch.randn(T, 2 * H * (D + E) + 3, generator=g).to(dt).cuda()
    a_raw, bias, w = torch.randn(T, H * D, generator=g).to(dt).cuda(), torch.randn(H * D, generator=g).cuda(), torch.randn(E, generator=g).cuda()
    one = torch.randn(8, H, D, E, generator=g).cuda()
    two = one.clone()
    y = hk.gla_norm(proj, a_raw, (H, D, E), bias, 16.0, w, one, *lay, 1e-6, dt)
    q, k, v, gate = proj[:, :2 * H * (D + E)].split([H * D, H * D, H * E, H * E], -1)
    o = hk.gla_scan(q.view(T, H, D), k.view(T, H, D), v.view(T, H, E), a_raw, bias, 16.0, two, *lay)
    assert torch.equal(y, hk.gated_head_norm(o, w, gate, 1e-6, dt, "silu").view(T, H * E)) and torch.equal(one, two)
