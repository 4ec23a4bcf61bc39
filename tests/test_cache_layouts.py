"""What the dense attention calls take as a KV cache: any physical order of [block, token, kv_head, d], rows of d contiguous."""
import pytest
import torch

from minivllm_amd.ops import hip


@pytest.mark.parametrize("order", [(0, 1, 2, 3), (0, 2, 1, 3), (1, 0, 2, 3)])
def test_strides(order):
    cache = torch.empty([(5, 16, 2, 8)[i] for i in order]).permute([order.index(i) for i in range(4)])
    assert cache.shape == (5, 16, 2, 8) and hip._cache_strides(cache) == cache.stride()[:3]
    assert hip._cache_strides(cache.unsqueeze(-1)) == cache.stride()[:3]          # one element behind a row's values
    with pytest.raises(ValueError):
        hip._cache_strides(cache.transpose(1, 3))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_dimension_of_one_behind(dtype):
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(*n, generator=g).to(dtype).cuda() for n in ((2, 4, 64), (6, 16, 2, 64), (6, 16, 2, 64)))
    tables = torch.arange(6, dtype=torch.int32, device="cuda").view(2, 3)
    lens, cu_q, cu_k = (torch.tensor(n, dtype=torch.int32, device="cuda") for n in ([40, 7], [0, 1, 2], [0, 40, 47]))
    for call in (lambda k, v: hip.paged_attention_decode(q, k, v, tables, lens, 0.125, 40),
                 lambda k, v: hip.paged_attention_prefill(q, k, v, cu_q, cu_k, tables, 0.125, 1)):
        assert torch.equal(call(k, v), call(k.unsqueeze(-1), v.unsqueeze(-1)))
