"""Which kernel of the hybrid library takes a call: the library's own rules, by sizes, strides and addresses."""
import pytest

from minivllm_amd.ops import hip_hybrid as hk

AT = 1 << 20                                           # an address of whole runs


@pytest.mark.parametrize("D,E,v_stride,shift,q_row,form", [
    # whole runs everywhere; whole key rows alone: the score products of the 16-bit instruction; neither
    (128, 128, 128, 0, 2048, 2), (128, 100, 100, 0, 2048, 1), (64, 20, 20, 0, 512, 1), (64, 64, 68, 0, 512, 1),
    (36, 64, 64, 0, 512, 0), (24, 20, 20, 0, 512, 0), (128, 100, 100, 2, 2048, 0), (128, 100, 100, 0, 2052, 0)])
def test_prompt_attention(D, E, v_stride, shift, q_row, form):
    a = (AT + shift, q_row, D, AT, AT, AT, 8, 1024, D, E, v_stride)
    assert hk._tiles_form(*a, 0) == form
    # float rows: the kernels of whole runs or the general one
    assert hk._tiles_form(*a, 2) == (2 if form == 2 else 0)
    # a value cache or an output off 16 bytes takes nothing from the score products
    if form == 2:
        assert hk._tiles_form(*a[:4], AT + 2, *a[5:], 0) == 1 and hk._tiles_form(*a[:5], AT + 2, *a[6:], 0) == 1
