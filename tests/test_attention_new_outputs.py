"""Attention into new outputs (``clear``): rows that no sequence owns become zeros, the others hold what they would
without it, whichever kernel runs; without ``clear`` foreign rows stay as they are."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,E,form", [(64, 64, 2), (128, 40, 2), (48, 36, 1), (160, 160, 0)])
@pytest.mark.parametrize("ahead,behind,qlens", [(0, 0, [5, 130]), (2, 3, [1, 64, 0, 129]), (1, 300, [40]), (0, 7, [0, 0])])
def test_prompt_rows(dtype, D, E, form, ahead, behind, qlens):
    from minivllm_amd.ops import hip_hybrid as hk
    torch.manual_seed(D)
    H, G, bs, B = 4, 2, 32, len(qlens)
    T, own = ahead + sum(qlens) + behind, sum(qlens)
    pages = [-(-max(n, 1) // bs) for n in qlens]
    tables = torch.arange(B * max(pages), dtype=torch.int32, device="cuda").view(B, -1)
    kc, vc = (torch.randn(tables.numel(), bs, G, n, device="cuda").to(dtype) for n in (D, E))
    q = torch.randn(T, H, D, device="cuda").to(dtype)
    cu = torch.tensor([ahead] + (ahead + torch.tensor(qlens).cumsum(0)).tolist(), dtype=torch.int32, device="cuda")
    pos, row_seq = torch.zeros(T, dtype=torch.int32), torch.full((T,), -1, dtype=torch.int32)
    at = ahead
    for b, n in enumerate(qlens):
        pos[at:at + n], row_seq[at:at + n] = torch.arange(n), ahead + b
        at += n
    got = []
    for clear in (True, False):
        out = torch.full((T, H, E), float("nan"), dtype=dtype, device="cuda")
        hk.sink_attention_prefill(q, kc, vc, cu, cu, tables, 0.1, None, None, out, positions=pos.cuda(), max_q=max(qlens),
                                  row_seq=row_seq.cuda(), first_seq=ahead, clear=clear)
        got.append(out)
    new, old = got
    assert torch.equal(new[ahead:ahead + own], old[ahead:ahead + own]) and torch.isfinite(new[ahead:ahead + own]).all()
    assert not new[ahead + own:].any() and torch.isnan(new[:ahead]).all()        # (rows ahead are another call's)
    assert torch.isnan(old[:ahead]).all() and torch.isnan(old[ahead + own:]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,E", [(64, 64), (128, 128), (48, 40)])
def test_next_token_rows(dtype, D, E):
    from minivllm_amd.ops import hip_hybrid as hk
    torch.manual_seed(E)
    H, G, bs, lens = 4, 2, 16, [0, 17, 0, 300, 1, 0]
    tables = torch.arange(6 * 19, dtype=torch.int32, device="cuda").view(6, 19)
    kc, vc = (torch.randn(6 * 19, bs, G, n, device="cuda").to(dtype) for n in (D, E))
    q, ctx = torch.randn(6, H, D, device="cuda").to(dtype), torch.tensor(lens, dtype=torch.int32, device="cuda")
    got = []
    for clear in (True, False):
        out = torch.full((6, H, E), float("nan"), dtype=dtype, device="cuda")
        hk.sink_attention_decode(q, kc, vc, tables, ctx, 0.1, None, None, out, 300, clear=clear)
        got.append(out)
    for b, n in enumerate(lens):
        if n:
            assert torch.equal(got[0][b], got[1][b]) and torch.isfinite(got[0][b]).all()
        else:
            assert not got[0][b].any() and torch.isnan(got[1][b]).all()
