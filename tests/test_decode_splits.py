"""Context splits of a decode step: the host asks for as many as the kernel uses for the longest context."""
import gc
import weakref

import numpy as np
import pytest
import torch

from minivllm_amd.ops import hip


def _in_use(tiles, splits, waves):
    """``splits_in_use`` of csrc/attn_decode.hip."""
    if tiles <= waves + waves // 4:
        return 1
    return min(splits, max(min(8, -(-2 * tiles // waves)), -(-tiles // waves)))


@pytest.mark.parametrize("kv_heads", [1, 2, 3, 4, 8])
def test_no_split_is_left_unused(kv_heads):
    for batch in range(1, 300):
        for context in (0, 1, 160, 161, 300, 320, 321, 385, 512, 513, 1025, 2048, 4096, 32768):
            n = hip.decode_num_splits(batch, kv_heads, context)
            waves = 8 if n * kv_heads * batch <= 256 else 4               # (the launcher's rule)
            assert n == _in_use(-(-context // 32), n, waves) <= 32, (batch, context, n)
            assert n <= hip.decode_num_splits(batch, kv_heads, None)


def test_a_growing_context_is_worked_out_once_per_tile():
    hip._splits_of.cache_clear()
    for context in range(1, 1025):
        hip.decode_num_splits(1, 8, context)
    assert hip._splits_of.cache_info().misses == 1024 // 32


@pytest.mark.parametrize("number", [np.int64, np.array, torch.tensor])
def test_context_of_any_whole_number(number):
    """What was accepted as a length stays so: numbers of numpy and tensors of one element, which are read at each call and not kept."""
    context = number(512)
    kept = weakref.ref(context) if torch.is_tensor(context) else None
    for length in (512, 4096, 100):
        if kept:
            context.fill_(length)
        else:
            context = number(length)
        assert hip.decode_num_splits(1, 8, context) == hip.decode_num_splits(1, 8, length)
    del context
    gc.collect()
    assert not kept or kept() is None
