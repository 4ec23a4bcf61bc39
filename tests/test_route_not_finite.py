"""Routers over rows that are not numbers (rows of no sequence may hold anything): what they choose stays inside their own row."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from minivllm_amd.ops import hip_hybrid as hk


@pytest.mark.parametrize("score,groups,keep", [("softmax", 4, 2), ("softmax", 1, 1), ("sigmoid", 4, 2), ("chosen", 1, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_beside_one_that_is_no_number(score, groups, keep, dtype):
    g = torch.Generator().manual_seed(groups)
    h, w = torch.randn(9, 64, generator=g).to(dtype).cuda(), torch.randn(8, 64, generator=g).cuda()
    bias = torch.zeros(8, device="cuda") if score == "chosen" else None
    want = hk.grouped_route(h, w, 3, groups, keep, score, bias)
    bad = h.clone()
    bad[[0, 4, 8], 5] = torch.tensor([float("nan"), float("nan"), float("inf")], dtype=dtype, device="cuda")
    for _ in range(3):
        got = hk.grouped_route(bad, w, 3, groups, keep, score, bias)
        rows = [1, 2, 3, 5, 6, 7]
        assert torch.equal(got[rows], want[rows])
        if score != "chosen":
            assert not got[4].any()                        # (no score of the row is a number)
