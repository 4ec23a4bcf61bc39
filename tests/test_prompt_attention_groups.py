"""Prompt attention: groups of waves that share out the key tiles of a workgroup's queries.  Launches on both sides of the lines between the forms, against float64: contexts of fewer tiles than there are groups, of as many,
of one more; windows and kept first keys that leave a group without a tile; an infinity beside finite rows."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from minivllm_amd.ops import hip_hybrid as hk


def _exact(q, k, v, past, scale, window, keep, sink):
    n, H, _ = q.shape
    r = H // k.shape[1]
    kt, vt = (x.double().transpose(0, 1).repeat_interleave(r, 0) for x in (k, v))
    z = torch.matmul(q.double().transpose(0, 1), kt.transpose(1, 2)) * scale
    i, j = torch.arange(past, past + n)[:, None], torch.arange(k.shape[0])[None]
    off = j > i
    if window:
        off = off | ((i - j >= window) & (j >= keep))
    z = z.masked_fill(off.to(z.device), -math.inf)
    z = torch.cat([z, sink.double()[:, None, None].expand(H, n, 1)], -1)
    return torch.matmul(z.softmax(-1)[..., :-1], vt).transpose(0, 1)


@pytest.mark.parametrize("D,E", [(64, 64), (128, 64), (48, 40), (128, 128), (72, 128)])
@pytest.mark.parametrize("H", [4, 48])                      # 40 .. 44 and 480 .. 528 tiles of 128 queries
@pytest.mark.parametrize("window,keep", [(0, 0), (40, 5), (130, 0)])
@pytest.mark.parametrize("dt,bs", [(torch.float32, 32), (torch.bfloat16, 64), (torch.bfloat16, 16)])
def test_forms(D, E, H, window, keep, dt, bs):
    g = torch.Generator().manual_seed(D + E + H)
    new, past = [1, 31, 33, 64, 65, 127, 129, 300], [0, 0, 95, 0, 64, 1, 200, 33]
    G, total = 2, [n + p for n, p in zip(new, past)]
    pages = [-(-n // bs) for n in total]
    perm, tables, at = torch.randperm(sum(pages), generator=g).int(), torch.zeros(len(new), max(pages), dtype=torch.int32), 0
    for b, n in enumerate(pages):
        tables[b, :n] = perm[at:at + n]
        at += n
    kc, vc = (torch.randn(sum(pages), bs, G, n, generator=g).to(dt) for n in (D, E))
    T = sum(new)
    q, sink, scale = torch.randn(T, H, D, generator=g).to(dt), torch.randn(H, generator=g), D ** -0.5
    cu = torch.tensor([0] + new).cumsum(0).int()
    cu_k = torch.tensor([0] + total).cumsum(0).int()
    pos = torch.cat([torch.arange(p, p + n) for n, p in zip(new, past)]).int()
    bad = int(tables[7, 200 // bs]), 200 % bs               # a key of the last sequence that its late queries see
    for broken in (False, True):
        if broken:
            vc[bad[0], bad[1], 1, 3] = math.inf
        out = torch.empty(T, H, E, dtype=dt, device="cuda")
        hk.sink_attention_prefill(q.cuda(), kc.cuda(), vc.cuda(), cu.cuda(), cu_k.cuda(), tables.cuda(), scale, sink.cuda(), None,
                                  out, positions=pos.cuda(), max_q=max(new), row_seq=None, window=window, keep_first=keep)
        at = 0
        for b, (n, p) in enumerate(zip(new, past)):
            rows = tables[b].long()
            k, v = (c[rows].reshape(-1, G, c.shape[3])[:n + p].cuda() for c in (kc, vc))
            want = _exact(q[at:at + n].cuda(), k, v, p, scale, window, keep, sink.cuda())
            got = out[at:at + n].double()
            if broken and b == 7:
                i = torch.arange(p, p + n, device="cuda")
                sees = (i >= 200) & ((i - 200 < window) | (window == 0) | (200 < keep))
                assert torch.equal(got[:, H // 2:, 3].isinf(), sees[:, None].expand(n, H // 2))
                keep_cols = [e for e in range(E) if e != 3]
                got, want = got[..., keep_cols], want[..., keep_cols]
            # fp32 sums of up to 333 terms and exponentials of fp32 differences; the result in its type
            assert float((got - want).norm() / want.norm()) < (1e-6 if dt == torch.float32 else 2.0 ** -8), (b, broken)
            at += n


@pytest.mark.parametrize("D,E", [(64, 64), (128, 64), (128, 128), (64, 256), (256, 64), (256, 128)])
@pytest.mark.parametrize("H", [2, 32, 96])
@pytest.mark.parametrize("new,past", [([1, 33, 129, 300], [700, 0, 95, 900]), ([96, 65, 31, 1, 64, 96, 80], [0] * 7)])
@pytest.mark.parametrize("window", [0, 300])
@pytest.mark.parametrize("dt,bs", [(torch.float32, 32), (torch.bfloat16, 64), (torch.bfloat16, 16)])
def test_long_and_short_walks(D, E, H, new, past, window, dt, bs):
    if dt == torch.float32 and max(D, E) > 128:
        pytest.skip("float rows of more than 128 have another kernel")
    g = torch.Generator().manual_seed(D + E + H)
    G, total = 2, [n + p for n, p in zip(new, past)]
    pages = [-(-n // bs) for n in total]
    perm, tables, at = torch.randperm(sum(pages), generator=g).int(), torch.zeros(len(new), max(pages), dtype=torch.int32), 0
    for b, n in enumerate(pages):
        tables[b, :n] = perm[at:at + n]
        at += n
    kc, vc = (torch.randn(sum(pages), bs, G, n, generator=g).to(dt).cuda() for n in (D, E))
    T = sum(new)
    q, sink, scale = torch.randn(T, H, D, generator=g).to(dt).cuda(), torch.randn(H, generator=g).cuda(), D ** -0.5
    cu, cu_k = (torch.tensor([0] + x).cumsum(0).int().cuda() for x in (new, total))
    pos = torch.cat([torch.arange(p, p + n) for n, p in zip(new, past)]).int().cuda()
    out = torch.full((T, H, E), 7.0, dtype=dt, device="cuda")
    hk.sink_attention_prefill(q, kc, vc, cu, cu_k, tables.cuda(), scale, sink, None, out, positions=pos, max_q=max(new),
                              row_seq=None, window=window)
    at = 0
    for b, (n, p) in enumerate(zip(new, past)):
        rows = tables[b].long().cuda()
        k, v = (c[rows].reshape(-1, G, c.shape[3])[:n + p] for c in (kc, vc))
        want, got = _exact(q[at:at + n], k, v, p, scale, window, 0, sink), out[at:at + n].double()
        # fp32 sums of up to 1200 terms and exponentials of fp32 differences; the result in its type
        assert float((got - want).norm() / want.norm()) < (1e-6 if dt == torch.float32 else 2.0 ** -8), b
        at += n
