"""Next tokens on the matrix cores: contexts at the edges of tiles, of waves and of splits, groups of heads that do not fill
sixteen columns, windows that leave waves or splits without a tile, rows without a sequence, infinities; against float64."""
import math

import pytest
import torch

from minivllm_amd.ops import hip_hybrid as hk


@pytest.mark.parametrize("batch,kv_heads,heads,seen,splits", [
    (1, 8, 16, 512, 1), (1, 8, 16, 513, 2), (1, 8, 16, 8192, 16), (4, 8, 16, 1024, 2), (16, 8, 16, 4096, 2), (32, 8, 16, 4096, 2),
    (64, 8, 16, 2048, 1), (1, 1, 17, 513, 2), (128, 1, 32, 4096, 2), (64, 8, 16, 8192, 4), (65, 8, 16, 8192, 3), (1, 8, 16, None, 2)])
def test_splits(batch, kv_heads, heads, seen, splits):
    assert hk.next_splits(batch, kv_heads, heads, seen) == splits


@pytest.mark.parametrize("groups,R,width,seen,matrix", [
    (512, 2, 256, 1024, True), (1023, 1, 256, 129, True), (1024, 1, 256, 129, False), (2047, 2, 256, 128, True), (2048, 2, 256, 128, False), (1024, 2, 256, 1536, False), (1024, 2, 256, 1537, True),
    (1365, 1, 192, 200, True), (1366, 2, 192, 200, False), (2047, 3, 256, 16, True), (2048, 3, 256, 16, False), (2048, 4, 256, 17, True),
    (2048, 4, 128, 1, True), (8192, 5, 256, 1, True), (6143, 1, 128, 16, True), (6144, 2, 128, 64, False), (6144, 2, 128, 65, True),
    (8192, 1, 256, None, True), (8192, 1, 256, 0, True)])
def test_units(groups, R, width, seen, matrix):
    assert hk.next_pays(groups, R, width, seen) is matrix


def _exact(q, k, v, scale, lo, keep, slopes, sink, gate):
    r = q.shape[0] // k.shape[1]
    kt, vt = (x.double().transpose(0, 1).repeat_interleave(r, 0) for x in (k, v))
    n = k.shape[0]
    z = torch.matmul(kt, q.double()[:, :, None])[..., 0] * scale
    j = torch.arange(n, device=q.device)
    if slopes is not None:
        z = z - slopes.double()[:, None] * (n - 1 - j)
    seen = (j >= lo) | (j < keep)
    z, vt = z[:, seen], vt[:, seen]
    if sink is not None:
        z = torch.cat([z, sink.double()[:, None]], -1)
    p = z.softmax(-1)[:, :vt.shape[1]]
    o = torch.matmul(p[:, None], vt)[:, 0]
    return o if gate is None else o * gate.double().sigmoid()[:, None]


@pytest.mark.gpu
@pytest.mark.parametrize("D,E", [(128, 128), (64, 64), (128, 64), (64, 128)])
@pytest.mark.parametrize("G,R", [(2, 1), (1, 5), (2, 16), (1, 20), (48, 2)])    # (48: workgroups of four waves)
@pytest.mark.parametrize("rule", [{}, {"window": 40, "keep_first": 5}, {"window": 300}, {"chunk": 256}, {"slopes": True}])
@pytest.mark.parametrize("bs", [32, 12])
@pytest.mark.parametrize("matrix", [True, False])
def test_against_exact(D, E, G, R, rule, bs, matrix, monkeypatch):
    monkeypatch.setattr(hk, "next_pays", lambda *a: matrix)               # (the steps are too few for the vector units)
    lens = [1, 31, 0, 32, 33, 256, 257, 513, 0, 1025, 2100]
    dev, H, B = "cuda", G * R, len(lens)
    g = torch.Generator().manual_seed(D + E + G + R)
    pages = [-(-n // bs) for n in lens]
    tables, perm, at = torch.zeros(B, max(pages), dtype=torch.int32), torch.randperm(sum(pages), generator=g).int(), 0
    for b, n in enumerate(pages):
        tables[b, :n] = perm[at:at + n]
        at += n
    kc, vc = (torch.randn(sum(pages), bs, G, n, generator=g).bfloat16().to(dev) for n in (D, E))
    q = torch.randn(B, H * D + 8, generator=g).bfloat16().to(dev)[:, :H * D].unflatten(1, (H, D))     # rows further apart
    options = not rule or "window" in rule
    sink = torch.randn(H, generator=g).to(dev) if options else None
    gate = torch.randn(B, H + 3, generator=g).bfloat16().to(dev)[:, :H] if options else None
    slopes = (torch.rand(H, generator=g) * 0.1).to(dev) if "slopes" in rule else None
    window, keep, chunk = rule.get("window", 0), rule.get("keep_first", 0), rule.get("chunk", 0)
    ctx = torch.tensor(lens, dtype=torch.int32, device=dev)

    def call(clear):
        out = torch.full((B, H, E), 7.0, dtype=torch.bfloat16, device=dev)
        hk.sink_attention_decode(q, kc, vc, tables.to(dev), ctx, D ** -0.5, sink, gate, out, max_context_len=max(lens),
                                 window=window, keep_first=keep, slopes=slopes, chunk=chunk, clear=clear)
        return out

    def compare(out, skip=None):
        for b, n in enumerate(lens):
            if n == 0 or b == skip:
                continue
            rows = tables[b].long().to(dev)
            k, v = (c[rows].reshape(-1, G, c.shape[3])[:n] for c in (kc, vc))
            lo = max(0, n - window) if window else (n - 1) // chunk * chunk if chunk else 0
            want = _exact(q[b], k, v, D ** -0.5, lo, keep, slopes, sink, None if gate is None else gate[b])
            got = out[b].double()
            # fp32 sums of up to 2100 terms, then one rounding to bfloat16
            assert float((got - want).norm() / want.norm()) < 2.0 ** -8, (b, n)

    out = call(True)
    compare(out)
    assert not out[2].any() and not out[8].any()
    assert bool((call(False)[2] == 7.0).all())
    # an infinity in a key's value: that column alone, of the heads that see it; where nobody sees it, nothing
    where = lens[10] - 50
    page, row = int(tables[10, where // bs]), where % bs
    vc[page, row, G - 1, 3] = math.inf
    out = call(True)
    compare(out, skip=10)
    seen = not (window == 40 or (chunk and where < (lens[10] - 1) // chunk * chunk))
    bad = torch.zeros(H, E, dtype=torch.bool, device=dev)
    if seen:
        bad[H - R:, 3] = True
    if slopes is None:                # (a weight may come out as zero under a slope: then NaN or finite)
        assert torch.equal(~out[10].isfinite(), bad)
    else:
        assert bool(out[10][~bad].isfinite().all())
    kc[page, row, 0, 1] = math.nan
    out = call(True)
    compare(out, skip=10)
    if seen:
        assert bool(out[10, :R].isnan().all())
    else:
        compare(out)


@pytest.mark.gpu
@pytest.mark.parametrize("D,E,n", [(128, 128, 1024), (64, 64, 300), (128, 64, 700)])
@pytest.mark.parametrize("spread", [1.0, 2.0, 4.0])
def test_sums_are_no_further_from_float64_than_on_the_vector_units(D, E, n, spread):
    """The partial results of two splits, which are fp32, ahead of the rounding that hides what is below it."""
    dev, B, G, H, bs, S = "cuda", 8, 4, 8, 64, 2
    pages, ratios = -(-n // bs), []
    for seed in range(6):
        g = torch.Generator(device=dev).manual_seed(seed)
        kc, vc = (torch.randn(B * pages, bs, G, m, generator=g, device=dev).bfloat16() for m in (D, E))
        q = (spread * torch.randn(B, H, D, generator=g, device=dev)).bfloat16()
        sink = torch.randn(H, generator=g, device=dev)
        tables = torch.arange(B * pages, device=dev, dtype=torch.int32).view(B, pages)
        lens = torch.full((B,), n, dtype=torch.int32, device=dev)
        out = torch.empty(B, H, E, dtype=torch.bfloat16, device=dev)
        want = torch.stack([_exact(q[b], *(c[b * pages:(b + 1) * pages].reshape(-1, G, c.shape[3])[:n] for c in (kc, vc)),
                                   D ** -0.5, 0, 0, None, sink, None) for b in range(B)])
        err = []
        for launch, own, last in ((hk._nxa, [], []), (hk._split, hk._pool_args(kc, vc, E, H, None, 0.0, 0, None, None), [0])):
            ws = torch.zeros(B, H, S, E + 2, device=dev)
            hk._check(launch(q.data_ptr(), H * D, D, kc.data_ptr(), vc.data_ptr(), tables.data_ptr(), pages, bs, lens.data_ptr(),
                             sink.data_ptr(), None, 0, out.data_ptr(), ws.data_ptr(), D ** -0.5, B, H, G, D, E, S, 0, 0, None, E,
                             *own, 0, 0, *last, hk._stream()), "attention")
            m, l, o = ws[..., 0].double(), ws[..., 1].double(), ws[..., 2:].double()
            top = torch.maximum(m.amax(-1), sink.double())
            f = (m - top[..., None]).exp()
            err.append(((o * f[..., None]).sum(2) / ((l * f).sum(-1) + (sink.double() - top).exp())[..., None] - want).norm())
        ratios.append(math.log(float(err[0] / err[1])))
    # the mean of six; a tenth for their spread (single ones differ by up to a quarter)
    assert sum(ratios) / len(ratios) <= math.log(1.1), ratios
