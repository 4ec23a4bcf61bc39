"""Latent attention with many query rows and long value rows: two waves share each score product."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from minivllm_amd.ops import hip_hybrid as hk


@pytest.mark.parametrize("H,R,P,bs,window,lens,qlens", [
    # both widths of the key rows (one with columns to spare), pages of whole tiles and not, a window that
    # starts inside tiles; prompts of one row, of a part of a tile, behind a prefix
    (128, 512, 64, 32, 0, [90, 1, 130], [90, 1, 33]),
    (128, 512, 128, 16, 40, [90, 97, 64], [90, 64, 2]),
    (101, 264, 56, 12, 33, [115, 115, 40], [115, 3, 40]),
])
@pytest.mark.parametrize("with_sink", [False, True])
def test_pairs_of_waves(H, R, P, bs, window, lens, qlens, with_sink):
    assert len(lens) * -(-max(qlens) * H // 64) > 512                # (more than fit the card at once)
    torch.manual_seed(H + R)
    B, D, T, dt = len(lens), R + P, sum(qlens), torch.bfloat16
    pages = [-(-n // bs) for n in lens]
    tables, at = torch.zeros(B, max(pages), dtype=torch.int32), 0
    perm = torch.randperm(sum(pages))
    for b, n in enumerate(pages):
        tables[b, :n] = perm[at:at + n]
        at += n
    cache = torch.randn(sum(pages), bs, 1, D).to(dt)
    q_abs, q_rot = torch.randn(H, T, R).to(dt), torch.randn(T, H, P).to(dt)
    sink, scale = (2.0 * torch.randn(H) if with_sink else None), 1.5 * D ** -0.5
    cu_q = torch.tensor([0] + torch.tensor(qlens).cumsum(0).tolist(), dtype=torch.int32)
    pos = torch.cat([torch.arange(n - m, n) for n, m in zip(lens, qlens)]).to(torch.int32)
    got = torch.full((T, H, R), float("nan"), dtype=dt, device="cuda")
    hk.latent_attention_prefill(q_abs.cuda(), q_rot.cuda(), cache.cuda(), cu_q.cuda(), tables.cuda(), pos.cuda(), scale,
                                None if sink is None else sink.cuda(), got, max(qlens), window)
    for b in range(B):
        rows = cache[tables[b, :pages[b]].long()].reshape(-1, D)[:lens[b]].double()
        sl = slice(int(cu_q[b]), int(cu_q[b + 1]))
        q = torch.cat([q_abs[:, sl].transpose(0, 1), q_rot[sl]], -1).double()      # [n, H, D]
        s = torch.einsum("nhd,kd->hnk", q, rows) * scale
        back = pos[sl].long()[:, None] - torch.arange(lens[b])[None]
        s = s.masked_fill((back < 0) | ((back >= window) if window else False), float("-inf"))
        if with_sink:
            s = torch.cat([s, sink.double()[:, None, None].expand(H, s.shape[1], 1)], -1)
        w = s.softmax(-1)[..., :lens[b]]
        want = torch.einsum("hnk,kr->nhr", w, rows[:, :R])
        # the result is rounded to bfloat16, 8 significant bits (2^-8 of itself at most); weights keep 17 bits and sums 24 against values
        # below 6, scores err by D 2^-24 of the sum of |q k| scale (below 2 sqrt(D)): all below 2^-10
        bound = 2.0 ** -8 * want.abs() + 2.0 ** -10
        worst = ((got[sl].cpu().double() - want).abs() / bound).max()
        assert float(worst) <= 1.0, (b, float(worst))
