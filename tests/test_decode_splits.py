"""Context splits of a decode step: the host asks for as many as the kernel uses for the longest context."""
import pytest

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
