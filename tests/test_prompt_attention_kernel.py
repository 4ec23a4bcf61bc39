"""Prompt portions over bfloat16 and float caches (``csrc/hybrid/hybrid_prompts.hip``) against the plain form in
fp32 on CPU copies: head sizes at the edges of the instances, pages smaller and larger than a key
tile, portions around a wave's and a workgroup's queries, every option; and the operands that the
general tile kernel takes instead."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from minivllm_amd.ops import hip_hybrid as hk
from minivllm_amd.ops import torch_seqmix as ref

LENS = [1, 31, 33, 64, 65, 127, 129, 300]          # contexts
PORTIONS = [1, 31, 2, 64, 33, 127, 129, 200]       # their last tokens are this step's


def close(got, want, top):
    """Both round the same sum (to bfloat16, whose numbers lie up to 2^-7 of their size apart: one step of it),
    and the fp32 sums of up to 300 products of weights (their sum 1) with values <= ``top`` differ themselves: scores
    of up to 128 (256) products err by a few 2^-22, weights by that of themselves.  The bits are tested below."""
    step = 2.0 ** -7 if got.dtype == torch.bfloat16 else 0.0
    got, want = got.float(), want.float()
    d = (got - want).abs()
    assert bool((d <= step * torch.maximum(got.abs(), want.abs()) + 2.0 ** -19 * top).all()), float(d.max())


def step(G, D, E, bs, seed=0, pooled=0, dt=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    need = [-(-n // bs) for n in LENS]
    ids = torch.randperm(sum(need), generator=g).int()
    tables = torch.zeros(len(LENS), max(need) + 1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(need):
        tables[b, :n] = ids[at:at + n]
        at += n
    rows = sum(need) * bs
    extra = sum(need) * -(-bs // pooled) if pooled else 0
    k, v = (torch.randn((rows + extra) * G, n, generator=g).to(dt) for n in (D, E))
    cu_q = torch.tensor([0] + PORTIONS).cumsum(0).int()
    cu_k = torch.tensor([0] + LENS).cumsum(0).int()
    pos = torch.cat([torch.arange(L - n, L) for L, n in zip(LENS, PORTIONS)]).int()
    return g, k, v, rows, tables, cu_q, cu_k, pos


def caches(k, v, rows, G, D, E, bs, pooled):
    n = rows // bs
    kc, vc = k[:rows * G].view(n, bs, G, D), v[:rows * G].view(n, bs, G, E)
    if not pooled:
        return kc, vc, None, None
    pr = -(-bs // pooled)
    return kc, vc, k[rows * G:].view(n, pr, G, D), v[rows * G:].view(n, pr, G, E)


OPTIONS = [dict(), dict(window=40, keep_first=5), dict(chunk=48), dict(slopes=True),
           dict(window=33, pool=8, temps=True, softcap=5.0)]


def compare(H, G, D, E, bs, opt, dt, shift=0):
    """The kernel that takes these operands (q ``shift`` numbers off 16 bytes) against the plain form."""
    opt = dict(opt)
    pool = opt.get("pool", 0)
    g, k, v, rows, tables, cu_q, cu_k, pos = step(G, D, E, bs, pooled=pool, dt=dt)
    T = int(cu_q[-1])
    proj = torch.randn(T, H * D + H, generator=g).to(dt)
    q, gate = proj[:, :H * D].view(T, H, D), proj[:, H * D:]
    sink = torch.randn(H, generator=g) if opt.get("softcap") or not opt else None
    if opt.pop("slopes", None):
        opt["slopes"] = torch.rand(H, generator=g) * 0.2
    if opt.pop("temps", None):
        opt["temps"] = torch.randn(H, generator=g)
    if H % 8 or shift:                                   # q rows of whole 16-byte runs only with H % 8 == 0
        q = q.contiguous()

    def call(f, to, q, **kw):
        kc, vc, kp, vp = caches(to(k), to(v), rows, G, D, E, bs, pool)
        o = {n: to(x) if torch.is_tensor(x) else x for n, x in opt.items()}
        if pool:
            o.update(k_pool=kp, v_pool=vp)
        return f(q, kc, vc, to(cu_q), to(cu_k), to(tables), D ** -0.5, None if sink is None else to(sink),
                 to(gate), to(torch.zeros(T, H, E, dtype=dt)), **kw, **o)

    want = call(ref.sink_attention_prefill, lambda x: x, q)
    gq = q.cuda()
    if shift:
        gq = torch.empty(q.numel() + shift, dtype=dt, device="cuda")[shift:].view(q.shape).copy_(q)
    got = call(hk.sink_attention_prefill, lambda x: x.cuda(), gq, positions=pos.cuda(), max_q=max(PORTIONS)).cpu()
    close(got, want, float(v.abs().max()))


@pytest.mark.parametrize("H,G,D,E", [(2, 1, 128, 128), (8, 4, 64, 64), (16, 2, 8, 16), (3, 3, 72, 136), (2, 2, 256, 120),
                                     (1, 1, 40, 256), (4, 2, 136, 64), (2, 1, 128, 256)])
@pytest.mark.parametrize("bs", [16, 64, 128])
@pytest.mark.parametrize("opt", OPTIONS)
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_every_instance_and_option(H, G, D, E, bs, opt, dt):
    compare(H, G, D, E, bs, opt, dt)


@pytest.mark.parametrize("bs", [1, 4, 8, 12, 24, 32, 40, 96])
@pytest.mark.parametrize("opt", [dict(), dict(window=40, keep_first=37), dict(window=70)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_pages_of_every_kind(bs, opt, dt):
    """Pages of whole tiles of 32 (one descriptor a tile), of whole runs of eight (one a piece) and of neither (every row
    looked up), powers of two or not, kept first keys that end inside a tile."""
    compare(4, 2, 128, 64, bs, opt, dt)


@pytest.mark.parametrize("H,G,D,E,shift", [(4, 2, 128, 100, 0), (8, 4, 64, 20, 0), (3, 1, 144, 36, 0),    # whole key rows
                                           (4, 2, 36, 64, 0), (2, 1, 64, 64, 1), (2, 2, 128, 128, 3)])    # neither
@pytest.mark.parametrize("opt", OPTIONS)
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_every_option_of_the_general_kernel(H, G, D, E, shift, opt, dt):
    compare(H, G, D, E, 64, opt, dt, shift)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,E,shift", [(64, 64, 1), (36, 64, 0), (64, 20, 0), (128, 128, 2)])
def test_operands_of_the_general_kernel(D, E, shift, dt):
    """Odd sizes and addresses stay with the kernel that takes any: same results."""
    H, G, bs = 4, 2, 64
    g, k, v, rows, tables, cu_q, cu_k, pos = step(G, D, E, bs, dt=dt)
    T = int(cu_q[-1])
    flat = torch.randn(T * H * D + shift, generator=g).to(dt)
    kc, vc, _, _ = caches(k, v, rows, G, D, E, bs, 0)
    out = torch.zeros(T, H, E, dtype=dt)
    want = ref.sink_attention_prefill(flat[shift:].view(T, H, D), kc, vc, cu_q, cu_k, tables, D ** -0.5, None, None, out)
    got = hk.sink_attention_prefill(flat.cuda()[shift:].view(T, H, D), kc.cuda(), vc.cuda(), cu_q.cuda(), cu_k.cuda(),
                                    tables.cuda(), D ** -0.5, None, None, torch.zeros_like(out).cuda(),
                                    positions=pos.cuda(), max_q=max(PORTIONS)).cpu()
    close(got, want, float(v.abs().max()))


def test_values_inside_the_key_rows():
    H, G, D, E, bs = 2, 1, 128, 64, 64
    g, k, _, rows, tables, cu_q, cu_k, pos = step(G, D, E, bs)
    T = int(cu_q[-1])
    kc = k[:rows].view(-1, bs, G, D)
    q = torch.randn(T, H, D, generator=g).bfloat16()
    want = ref.sink_attention_prefill(q, kc, kc[..., :E], cu_q, cu_k, tables, D ** -0.5, None, None,
                                      torch.zeros(T, H, E, dtype=torch.bfloat16))
    kg = kc.cuda()
    got = hk.sink_attention_prefill(q.cuda(), kg, kg[..., :E], cu_q.cuda(), cu_k.cuda(), tables.cuda(), D ** -0.5, None,
                                    None, torch.zeros(T, H, E, dtype=torch.bfloat16).cuda(), positions=pos.cuda(),
                                    max_q=max(PORTIONS)).cpu()
    close(got, want, float(k.abs().max()))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,E,bs", [(128, 128, 64), (40, 72, 64), (64, 64, 16)])
@pytest.mark.parametrize("opt", [dict(), dict(window=40, keep_first=5)])
def test_infinities_stay_where_they_are(D, E, bs, dt, opt):
    """A key of infinity has no weight where its score is -infinity; a value of infinity makes its column of the rows
    that see it infinite; what is not a number makes the rows (key) or entries (value) that see it so; no other
    entry changes (float64, over the keys that a row sees)."""
    H, G, inf = 4, 2, float("inf")
    g, k, v, rows, tables, cu_q, cu_k, pos = step(G, D, E, bs, dt=dt)
    kc, vc, _, _ = caches(k, v, rows, G, D, E, bs, 0)

    def put(cache, b, j, head, column, x):
        cache[tables[b, j // bs], j % bs, head, column] = x

    put(kc, 2, 32, 0, 1, inf)                            # (sequence, key): the last key, one of a tile's middle, the first
    put(kc, 5, 70, 1, D - 1, -inf)
    put(kc, 7, 0, 0, 9, inf)
    put(kc, 7, 250, 1, 0, float("nan"))
    put(vc, 4, 40, 0, 3, -inf)
    put(vc, 6, 3, 1, E - 1, inf)
    put(vc, 6, 100, 0, 0, float("nan"))
    T = int(cu_q[-1])
    q = torch.randn(T, H, D, generator=g).to(dt)
    sink = torch.randn(H, generator=g)
    got = hk.sink_attention_prefill(q.cuda(), kc.cuda(), vc.cuda(), cu_q.cuda(), cu_k.cuda(), tables.cuda(), D ** -0.5,
                                    sink.cuda(), None, torch.zeros(T, H, E, dtype=dt).cuda(), positions=pos.cuda(),
                                    max_q=max(PORTIONS), **opt).cpu()
    want = torch.empty(T, H, E, dtype=torch.float64)
    for t in range(T):
        b, p = int(torch.searchsorted(cu_q[1:].contiguous(), t, right=True)), int(pos[t])
        lo = max(0, p - opt.get("window", p + 1) + 1)
        keys = list(range(min(opt.get("keep_first", 0), lo))) + list(range(lo, p + 1))
        at = [(int(tables[b, j // bs]), j % bs) for j in keys]
        kk, vv = (torch.stack([c[i, j] for i, j in at], 1).double() for c in (kc, vc))               # [G, keys, :]
        s = torch.einsum("hd,hnd->hn", q[t].double(), kk.repeat_interleave(H // G, 0)) * D ** -0.5
        s = torch.cat([s, sink.double()[:, None]], 1)
        w = torch.exp(s - s.max(1, keepdim=True)[0])
        w = (w / w.sum(1, keepdim=True))[:, :-1]
        x = w[:, :, None] * vv.repeat_interleave(H // G, 0)
        want[t] = torch.where((w > 0)[:, :, None] | w.isnan()[:, :, None], x, torch.zeros_like(x)).sum(1)
    assert int(want.isnan().any(2).sum()) > 20 and int(want.isinf().any(2).sum()) > 20
    assert bool(want.isfinite().all(2).sum() > T * H // 3)
    tol = dict(rtol=2 ** -7, atol=1e-5) if dt == torch.bfloat16 else dict(rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(got.double(), want, equal_nan=True, **tol)


@pytest.mark.parametrize("H,G,D,E", [(4, 2, 128, 128), (8, 4, 64, 64), (2, 1, 72, 40), (2, 2, 64, 128)])
@pytest.mark.parametrize("window", [0, 100])
def test_bits_over_float_caches(H, G, D, E, window):
    """Operands in parts lose nothing against the fp32 instruction: the same numbers through the kernel for whole
    runs and, queries off 16 bytes, through the general one; errors in the mean, counted from float64 (a tenth for
    the sample's own spread).  Operands of two parts would be 2^-17 off, a hundred times the general kernel's error."""
    bs = 64
    g, k, v, rows, tables, cu_q, cu_k, pos = step(G, D, E, bs, dt=torch.float32)
    kc, vc, _, _ = caches(k, v, rows, G, D, E, bs, 0)
    T = int(cu_q[-1])
    q = torch.randn(T, H, D, generator=g)
    want = torch.empty(T, H, E, dtype=torch.float64)
    for b, n in enumerate(LENS):
        rows_of = slice(int(cu_q[b]), int(cu_q[b + 1]))
        kk, vv = (c[tables[b, :-(-n // bs)].long()].reshape(-1, G, c.shape[3])[:n].double().repeat_interleave(H // G, 1)
                  for c in (kc, vc))
        z = torch.einsum("thd,nhd->htn", q[rows_of].double(), kk) * float(torch.tensor(D ** -0.5))
        back = pos[rows_of].long()[:, None] - torch.arange(n)[None]
        z = z.masked_fill((back < 0) | ((back >= window) if window else False), float("-inf"))
        want[rows_of] = torch.einsum("htn,nhe->the", z.softmax(-1), vv)
    err = []
    for shift in (0, 1):
        gq = torch.empty(q.numel() + shift, device="cuda")[shift:].view(q.shape).copy_(q)
        got = hk.sink_attention_prefill(gq, kc.cuda(), vc.cuda(), cu_q.cuda(), cu_k.cuda(), tables.cuda(), D ** -0.5, None,
                                        None, torch.zeros(T, H, E).cuda(), positions=pos.cuda(), max_q=max(PORTIONS),
                                        window=window).cpu()
        err.append(float((got.double() - want).norm() / want.norm()))
    assert err[0] <= 1.1 * err[1] and err[1] < 1e-6, err


def test_bits_of_the_weights_over_bfloat16_caches():
    """Weights keep 24 bits, which a bfloat16 result hides unless it is small against its terms: four keys whose
    values are chosen (in float64, key after key) so that the weighted sum all but vanishes.  fp32 scores below 4 and
    weights err by a few 2^-24 each; weights of 16 bits would by 2^-17."""
    H, D, E, bs, n = 8, 64, 64, 64, 4
    g = torch.Generator().manual_seed(5)
    q = torch.randn(1, H, D, generator=g).bfloat16()
    kc, vc = torch.zeros(1, bs, H, D).bfloat16(), torch.zeros(1, bs, H, E).bfloat16()
    kc[0, :n] = torch.randn(n, H, D, generator=g).bfloat16()
    w = torch.softmax(torch.einsum("hd,nhd->hn", q[0].double(), kc[0, :n].double()) * D ** -0.5, 1)
    order = w.argsort(1, descending=True)              # each value takes off what is left, the lightest key last
    left = torch.zeros(H, E, dtype=torch.float64)
    for i in range(n):
        h, j = torch.arange(H), order[:, i]
        v = (1 + torch.rand(H, E, generator=g)).bfloat16() if i == 0 else (-left / w[h, j][:, None]).bfloat16()
        vc[0, j, h] = v
        left = left + w[h, j][:, None] * v.double()
    assert float(left.abs().max()) < 2.0 ** -18
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32).cuda()                                   # noqa: E731
    got = hk.sink_attention_prefill(q.cuda(), kc.cuda(), vc.cuda(), i32(0, 1), i32(0, n), i32(0).view(1, 1), D ** -0.5, None,
                                    None, torch.zeros(1, H, E).bfloat16().cuda(), positions=i32(n - 1), max_q=1).cpu()
    assert float((got[0].double() - left).abs().max()) <= 2.0 ** -20
