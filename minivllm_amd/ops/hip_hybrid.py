"""Bindings for ``_hip_hybrid.so`` (``csrc/hybrid``): the gfx950 kernels of hybrid
decoders.  Same conventions as ``ops.hip``: raw device pointers, element strides, the current
HIP stream (so calls made during graph capture become graph nodes), no PyTorch fallback.  The
library is built on first use when it is missing (a few seconds, hipcc only).  Tensors are
bfloat16 or float32 (``dt`` 0 / 2); fp32 tensors (stream, state, router, norm weights) are always
fp32.  Function signatures mirror ``ops.torch_seqmix``.
"""
from __future__ import annotations

import ctypes
import functools
import os
from typing import Optional

import torch

from .native_call import bind

_LIB_PATH = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                         "_hip_hybrid.so")
if not os.path.exists(_LIB_PATH):
    from minivllm_amd import build as _build
    _build.build_hip_group("hybrid", verbose=False)
_lib = ctypes.CDLL(_LIB_PATH)

_L, _I, _F, _P = ctypes.c_long, ctypes.c_int, ctypes.c_float, ctypes.c_void_p


def _sig(name, *argtypes):
    return bind(_lib, name, argtypes)


_embed = _sig("hyb_embed_sum", _P, _P, _P, _P, _P, _L, _I, _F, _I, _P)
_norm = _sig("hyb_offset_rms_norm", _P, _P, _P, _L, _I, _F, _I, _P)
_post = _sig("hyb_post_norm_residual", _P, _L, _P, _F, _P, _P, _P, _P, _P, _L, _I, _F, _I, _P)
_rope = _sig("hyb_pair_rope_mix_store", _P, _P, _P, _L, _P, _P, _I, _P, _P, _I, _P, _P, _P, _L,
             _I, _I, _I, _I, _I, _P)
_ghn = _sig("hyb_gated_head_norm", _P, _P, _P, _L, _P, _L, _I, _I, _F, _I, _I, _I, _P)
_route = _sig("hyb_grouped_route", _P, _P, _P, _L, _I, _I, _I, _I, _I, _I, _I, _P)
_gelu = _sig("hyb_gelu_route_scale", _P, _P, _P, _L, _I, _I, _I, _P)
# head temperatures, soft cap, pool, pooled rows per page, first pooled row, chunk
_POOL = (_P, _F, _I, _I, _L, _I)
_attn = _sig("hyb_sink_attention_rows", _P, _L, _L, _P, _P, _P, _I, _I, _P, _P, _I, _P, _P, _L, _P,
             _F, _L, _I, _I, _I, _I, _I, _I, _I, _P, _I, *_POOL, _I, _P)
_tiles = _sig("hyb_sink_attention_tiles", _P, _L, _L, _P, _P, _P, _I, _I, _P, _P, _P, _P, _L, _P, _F,
              _I, _I, _I, _I, _I, _I, _I, _I, _I, _P, _I, *_POOL, _L, _L, _I, _P)
_tiles_ok = bind(_lib, "hyb_sink_attention_tiles_ok", [_I, _I], _I)
_f32_form = bind(_lib, "hyb_prompt_f32_form", [_I, _L, _I, _I, _I, _L], _I)
_prompt_groups = bind(_lib, "hyb_prompt_groups", [_I, _I, _L, _L], _I)
_longest_walk = bind(_lib, "hyb_prompt_longest_walk", [_I] * 5, _I)
_tiles_form = _sig("hyb_sink_attention_tiles_form", _P, _L, _L, _P, _P, _P, _I, _I, _I, _I, _I, _I)
_split = _sig("hyb_sink_attention_split", _P, _L, _L, _P, _P, _P, _I, _I, _P, _P, _P, _L, _P, _P, _F,
              _I, _I, _I, _I, _I, _I, _I, _I, _P, _I, *_POOL, _I, _I, _P)
_split_heads = _sig("hyb_sink_attention_split_heads", _I)
_split_ok = bind(_lib, "hyb_sink_attention_split_ok", [_I, _I], _I)
_nxa = _sig("hyb_next_attention", _P, _L, _L, _P, _P, _P, _I, _I, _P, _P, _P, _L, _P, _P, _F, _I, _I, _I, _I, _I, _I, _I, _I,
            _P, _I, _I, _I, _P)
_nxa_ok = bind(_lib, "hyb_next_attention_ok", [_I, _I], _I)
_prep = _sig("hyb_delta_prepare", _P, _L, _I, _P, _L, _I, _P, _I, _P, _I, _P, _P, _P, _P, _P, _P, _P,
             _P, _P, _P, _P, _P, _L, _I, _I, _I, _I, _I, _I, _P)
_prep_form = _sig("hyb_delta_prepare_form", _P, _L, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I)
_scan = _sig("hyb_delta_scan", _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _L, _I, _I, _I, _I, _I, _I, _P)
_scan_ws = bind(_lib, "hyb_delta_scan_ws", [_P, _P, _P, _P, _P, _L, _I, _I, _I, _I, _I], _L)
_next = _sig("hyb_delta_next", _P, _L, _I, _P, _L, _I, _P, _L, _P, _I, _P, _P, _P, _I, _P, _P, _P, _P, _P, _F, _I,
             _I, _I, _I, _I, _I, _I, _P)
_next_ok = bind(_lib, "hyb_delta_next_ok", [_I] * 5, _I)
_cscan = _sig("hyb_channel_delta_scan", _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _L, _I, _I, _I, _I, _I, _P)
_gla = _sig("hyb_gla_scan", _P, _P, _P, _L, _L, _L, _P, _L, _P, _F, _P, _P, _P, _P, _P, _L, _I, _I, _I, _I,
            _I, _P)
_mlstm = _sig("hyb_mlstm_scan", _P, _P, _P, _L, _L, _L, _P, _P, _L, _P, _P, _F, _P, _P, _P, _P, _P, _P,
              _P, _P, _L, _I, _I, _I, _I, _I, _P)
_mlstm_rows = _sig("hyb_mlstm_rows", _P, _L, _P, _P, _F, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _F, _L, _I, _I, _I, _I, _I, _P)
_gla_rows = _sig("hyb_gla_rows", _P, _L, _P, _L, _P, _F, _P, _P, _P, _P, _P, _P, _P, _I, _F, _L, _I, _I, _I, _I, _I, _P)
_mlstm_bytes = bind(_lib, "hyb_mlstm_chunks_bytes", [_P, _P, _P, _L, _L, _L, _L] + [_I] * 6, _L)
_chan = _sig("hyb_channel_chunks", _I, _P, _P, _P, _L, _L, _L, _P, _L, _P, _P, _F, _F, _P, _P, _P, _P, _P, _P, _P, _P, _L, _P,
             _I, _F, _I, _L, _I, _I, _I, _I, _I, _P)
_chan_bytes = bind(_lib, "hyb_channel_chunks_bytes", [_L] + [_I] * 8, _L)
_esin = _sig("hyb_embed_sinusoid", _P, _P, _P, _P, _P, _L, _I, _I, _P)
_rgn = _sig("hyb_residual_group_norm", _P, _P, _L, _P, _L, _P, _P, _L, _I, _I, _F, _I, _P)
_anm = _sig("hyb_add_normed_mean", _P, _P, _L, _P, _P, _L, _P, _L, _I, _F, _I, _P)
_uns = _sig("hyb_unit_norm_store", _P, _P, _L, _F, _P, _P, _P, _L, _I, _I, _I, _I, _P)
_swi = _sig("hyb_swiglu_route_scale", _P, _L, _P, _P, _L, _I, _I, _I, _I, _P)
_cap = _sig("hyb_tanh_cap", _P, _L, _F, _I, _P)
_rsn = _sig("hyb_residual_sum_norm", _P, _P, _P, _P, _I, _F, _P, _L, _I, _F, _I, _P)
_rnr = _sig("hyb_rms_norm_rows", _P, _L, _P, _P, _L, _I, _F, _I, _P)
_rns = _sig("hyb_row_norm_store", _P, _P, _P, _L, _P, _P, _F, _P, _P, _P, _L, _I, _I, _I, _I, _P)
_lrs = _sig("hyb_latent_rope_store", _P, _P, _L, _P, _L, _P, _F, _P, _P, _I, _P, _P, _P, _P, _L, _I,
            _I, _I, _I, _I, _F, _I, _P)
_xie = _sig("hyb_xielu", _P, _L, _P, _L, _I, _F, _F, _I, _P)
_ggn = _sig("hyb_gated_group_norm", _P, _P, _P, _P, _L, _P, _P, _L, _I, _I, _I, _F, _I, _P)
_sgt = _sig("hyb_sigmoid_gate", _P, _L, _L, _P, _L, _P, _L, _I, _I, _I, _P)
_hrs = _sig("hyb_half_rope_store", _P, _P, _P, _L, _P, _P, _I, _P, _P, _P, _P, _L, _I, _I, _I, _I, _I, _P)
_pbm = _sig("hyb_pool_block_means", _P, _P, _P, _P, _P, _P, _P, _I, _P, _L, _I, _I, _I, _I, _I, _I, _I, _P)
_utg = _sig("hyb_unturn_gate", _P, _L, _L, _P, _P, _P, _L, _P, _L, _I, _I, _I, _P)
_scv = _sig("hyb_short_conv", _P, _L, _P, _P, _P, _P, _P, _P, _P, _P, _L, _I, _I, _I, _I, _P)
_lru = _sig("hyb_rglru_scan", _P, _P, _P, _P, _P, _L, _P, _P, _P, _P, _P, _L, _I, _I, _I, _F, _I, _I, _P)
_crt = _sig("hyb_chosen_route", _P, _P, _P, _P, _L, _I, _I, _I, _I, _I, _P)
_cgl = _sig("hyb_capped_glu_route_scale", _P, _L, _P, _P, _L, _I, _I, _I, _I, _F, _F, _F, _I, _I, _P)
_hyp = _sig("hyb_hyper_update_norm", _P, _L, _L, _P, _P, _L, _P, _L, _P, _L, _P, _P, _P, _P, _P, _P, _P, _L, _I,
            _I, _I, _P)
_cor = _sig("hyb_corrected_route", _P, _P, _P, _P, _L, _I, _I, _I, _I, _F, _I, _P)
_gtg = _sig("hyb_gelu_tanh_glu", _P, _L, _P, _L, _I, _I, _P)

_cns = _sig("hyb_conv_norm_store", _P, _L, _P, _P, _P, _P, _F, _P, _P, _P, _P, _P, _P, _P, _P, _L, _I, _I, _I,
            _I, _I, _I, _I, _P)
_smx = _sig("hyb_shift_mix", _P, _P, _P, _P, _P, _P, _P, _P, _L, _I, _I, _I, _I, _P)
_rsq = _sig("hyb_relu_squared", _P, _L, _P, _L, _I, _I, _P)
_tgt = _sig("hyb_token_gate", _P, _L, _P, _P, _L, _L, _P, _L, _I, _I, _P)
_wkv = _sig("hyb_wkv_scan", _P, _P, _P, _L, _L, _L, _P, _L, _P, _P, _P, _P, _P, _P, _P, _L, _I, _I, _I, _I, _I, _P)
_lat = _sig("hyb_latent_attention", _P, _L, _L, _P, _L, _L, _P, _P, _I, _I, _P, _P, _P, _P, _P, _L, _L, _P,
            _F, _I, _I, _I, _I, _I, _I, _I, _P)
_latf = _sig("hyb_latent_formed_prompts", _P, _L, _L, _P, _L, _P, _P, _I, _I, _P, _P, _P, _P, _P, _P, _P, _L, _P,
             _F, _I, _I, _I, _I, _I, _I, _I, _I, _P)
_latr = _sig("hyb_latent_rows", _P, _L, _P, _L, _P, _F, _P, _P, _I, _I, _F, _P, _P, _P, _P, _P, _I, _I, _P, _P, _P, _P, _P, _F,
              _L, _I, _I, _I, _I, _I, _I, _I, _I, _I, _P)
_latr_ok = functools.lru_cache(maxsize=64)(bind(_lib, "hyb_latent_rows_ok", [_I] * 7, _I))
_latr_ws = bind(_lib, "hyb_latent_rows_ws", [_L, _I, _I, _I, _I], _L)
_latf_ok = functools.lru_cache(maxsize=64)(bind(_lib, "hyb_latent_formed_ok", [_I] * 6, _I))
_lat_ok = bind(_lib, "hyb_latent_attention_ok", [_I, _I], _I)

_DT = {torch.bfloat16: 0, torch.float32: 2}


def _dt(t: torch.Tensor) -> int:
    try:
        return _DT[t.dtype]
    except KeyError:
        raise TypeError(f"hybrid kernels take bfloat16 / float32 activations, got {t.dtype}")


def _stream() -> int:
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def _check(rc: int, name: str) -> None:
    if rc != 0:
        raise RuntimeError(f"{name} failed (code {rc}): shape outside the kernel's range or a "
                           f"HIP launch error")


def _ptr(t: Optional[torch.Tensor]) -> Optional[int]:
    return None if t is None else t.data_ptr()


def _f32(t: torch.Tensor) -> torch.Tensor:
    assert t.dtype == torch.float32 and t.is_contiguous(), "fp32 contiguous tensor expected"
    return t


def _i32(t: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    if t is None:
        return None
    assert t.dtype == torch.int32 and t.is_contiguous()
    return t


def _rows(t: torch.Tensor) -> int:
    """Row stride (elements) of a [T, ...] view whose trailing dims are dense."""
    assert t.stride(-1) == 1
    return t.stride(0) if t.shape[0] > 1 else int(t.stride(0) or t[0].numel())


# ------------------------------------------------------------------ embedding + norms
def embed_sum(ids, aux_rows, table, aux_table, scale=1.0):
    T, W = ids.shape[0], table.shape[1]
    x = torch.empty((T, W), dtype=torch.float32, device=table.device)
    _check(_embed(_ptr(_i32(ids)), _ptr(_i32(aux_rows)) if aux_table is not None else None,
                  table.data_ptr(), _ptr(aux_table), x.data_ptr(), T, W, float(scale), _dt(table), _stream()),
           "embed_sum")
    return x


def offset_rms_norm(x, w, eps, out_dtype):
    x = _f32(x)
    T, W = x.shape
    out = torch.empty((T, W), dtype=out_dtype, device=x.device)
    _check(_norm(x.data_ptr(), _f32(w).data_ptr(), out.data_ptr(), T, W, eps, _dt(out), _stream()),
           "offset_rms_norm")
    return out


def post_norm_residual(y, wb, x, eps, w_next, out_dtype, plain=False, raw=False, extra=None):
    x = _f32(x)
    T, W = x.shape
    assert y.shape == x.shape and y.stride(-1) == 1 and y.dtype == out_dtype and wb.numel() == W
    assert not (raw and w_next is not None)
    h = torch.empty((T, W), dtype=out_dtype, device=x.device) if raw or w_next is not None else None
    ids, table = extra if extra is not None else (None, None)
    if table is not None:
        assert table.is_contiguous() and table.shape[1] == W and table.dtype == y.dtype and ids.shape[0] >= T
    _check(_post(y.data_ptr(), _rows(y), _f32(wb).data_ptr(), 0.0 if plain else 1.0, _ptr(_i32(ids)),
                 _ptr(table), x.data_ptr(), _ptr(w_next), _ptr(h), T, W, eps, _dt(y), _stream()),
           "post_norm_residual")
    return h


# ------------------------------------------------------------------ rotation, value mix, store
def pair_rope_mix_store(q, k, v, positions, cos_sin, rot_dims, v_first, lam, v_mode,
                        k_cache, v_cache, slot_mapping):
    T, H, D = q.shape
    G, E = v.shape[1], v.shape[2]
    rs = q.stride(0)
    assert (T == 1 or (k.stride(0) == rs and v.stride(0) == rs)) and q.stride(1) == D \
        and k.stride(1) == D and v.stride(1) == E and q.stride(2) == 1, \
        "q / k / v must be views of one projection output"
    if k_cache is not None:
        assert k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.dtype == q.dtype
    if rot_dims:
        assert cos_sin.shape[1] == rot_dims and cos_sin.dtype == torch.float32
    if v_mode:
        assert v_first is not None and v_first.is_contiguous() and v_first.dtype == q.dtype \
            and v_first.numel() == T * G * E
    _check(_rope(q.data_ptr(), k.data_ptr(), v.data_ptr(), rs, _i32(positions).data_ptr(),
                 _ptr(cos_sin) if rot_dims else None, rot_dims, _ptr(v_first) if v_mode else None,
                 _f32(lam).data_ptr(), v_mode, _ptr(k_cache), _ptr(v_cache), _ptr(_i32(slot_mapping)),
                 T, H, G, D, E, _dt(q), _stream()), "pair_rope_mix_store")


# ------------------------------------------------------------------ attention with a sink
def _slopes(slopes, H):
    if slopes is None:
        return None
    assert slopes.dtype == torch.float32 and slopes.is_contiguous() and slopes.numel() == H
    return slopes.data_ptr()


def _value_rows(k_cache, v_cache):
    """Elements from one (slot, KV head) value row to the next.  The V cache is a dense tensor
    [blocks, block, G, E] or, when the values are stored inside the key rows, a view
    [blocks, block, G, E] of the leading E entries of each wider row."""
    n, bs, G, E = v_cache.shape
    vs = v_cache.stride(2) if G > 1 else v_cache.stride(1)
    assert v_cache.stride(3) == 1 and vs >= E and v_cache.stride(1) == G * vs \
        and (n == 1 or v_cache.stride(0) == bs * G * vs), "value rows must be evenly spaced"
    assert v_cache.dtype == k_cache.dtype and v_cache.shape[:3] == k_cache.shape[:3]
    return vs


def _pool_args(k_cache, v_cache, vs, H, temps, softcap, pool, k_pool, v_pool):
    """(temps, softcap, pool, pooled rows per page, first pooled row) for the attention kernels.
    The pooled caches lie behind the token caches in the same allocations, the same number of
    rows behind both."""
    tp = None
    if temps is not None:
        assert temps.dtype == torch.float32 and temps.is_contiguous() and temps.numel() == H
        tp = temps.data_ptr()
    if not pool:
        return tp, float(softcap), 0, 0, 0
    n, bs, G, D = k_cache.shape
    es = k_cache.element_size()
    assert k_pool.is_contiguous() and v_pool.is_contiguous() and k_pool.shape[0] == n \
        and k_pool.shape[2:] == (G, D) and v_pool.shape[:3] == k_pool.shape[:3] \
        and k_pool.shape[1] * pool >= bs and k_pool.dtype == k_cache.dtype
    base = (k_pool.data_ptr() - k_cache.data_ptr()) // (G * D * es)
    assert base > 0 and k_cache.data_ptr() + base * G * D * es == k_pool.data_ptr() \
        and v_cache.data_ptr() + base * G * vs * es == v_pool.data_ptr(), \
        "the pooled rows must follow their token cache in one allocation"
    return tp, float(softcap), int(pool), int(k_pool.shape[1]), int(base)


def _attention_rows(q, k_cache, v_cache, block_tables, row_seq, lens, len_add, scale, sink, gate, out,
                    seq_base=0, window=0, keep_first=0, slopes=None, temps=None, softcap=0.0, pool=0,
                    k_pool=None, v_pool=None, chunk=0):
    T, H, D = q.shape
    G, E = k_cache.shape[2], v_cache.shape[3]
    assert q.stride(2) == 1 and out.is_contiguous() and out.shape == (T, H, E) and out.dtype == q.dtype
    assert k_cache.is_contiguous() and k_cache.dtype == q.dtype
    vs = _value_rows(k_cache, v_cache)
    assert block_tables.dtype == torch.int32 and block_tables.stride(1) == 1
    if gate is not None:
        assert gate.stride(1) == 1 and gate.dtype == q.dtype
    _check(_attn(q.data_ptr(), q.stride(0), q.stride(1), k_cache.data_ptr(), v_cache.data_ptr(),
                 block_tables.data_ptr(), block_tables.stride(0), k_cache.shape[1],
                 _ptr(_i32(row_seq)), _i32(lens).data_ptr(), len_add,
                 _f32(sink).data_ptr() if sink is not None else None,
                 _ptr(gate), gate.stride(0) if gate is not None else 0, out.data_ptr(), scale, T,
                 H, G, D, E, seq_base, int(window), int(keep_first), _slopes(slopes, H), vs,
                 *_pool_args(k_cache, v_cache, vs, H, temps, softcap, pool, k_pool, v_pool), int(chunk), _dt(q),
                 _stream()), "sink_attention")
    return out


def sink_attention_step(q, k_cache, v_cache, block_tables, row_seq, positions, scale, sink, gate, out,
                        seq_base=0, window=0, keep_first=0, slopes=None, **pooled):
    """Rows of a prefill-form step, one workgroup per row: row t belongs to sequence
    ``row_seq[t]`` (< ``seq_base``: skipped), whose block table is row ``row_seq[t] - seq_base``
    of ``block_tables``, and sees ``positions[t] + 1`` keys."""
    return _attention_rows(q, k_cache, v_cache, block_tables, row_seq, positions, 1, scale, sink,
                           gate, out, seq_base, window, keep_first, slopes, **pooled)


def sink_attention_prefill(q, k_cache, v_cache, cu_q, cu_k, block_tables, scale, sink, gate, out,
                           positions=None, max_q=None, row_seq=None, first_seq=0,
                           window=0, keep_first=0, slopes=None, temps=None, softcap=0.0, pool=0,
                           k_pool=None, v_pool=None, chunk=0, clear=False):
    """The prompt portions of a step: sequence b owns rows cu_q[b] .. cu_q[b+1] (absolute rows
    of q / out / positions) and block table row b.  Runs the matrix-core tile kernel (fp32
    scores, weights and sums); head sizes it has no instance for go row by row.  ``cu_k`` is
    not needed (a row's context is its position + 1).  ``clear``: ``out`` is new, rows from
    ``first_seq`` on that none of the sequences owns become zeros (otherwise they stay as they are)."""
    T, H, D = q.shape
    G, E = k_cache.shape[2], v_cache.shape[3]
    nseq = cu_q.shape[0] - 1
    assert positions is not None, "the GPU form takes the rows' positions"
    if not _tiles_ok(D, E):
        assert row_seq is not None
        if clear:
            out[first_seq:].zero_()
        # ``first_seq``: number of the step's sequences ahead of these (its decode riders)
        return sink_attention_step(q, k_cache, v_cache, block_tables, row_seq, positions, scale,
                                   sink, gate, out, seq_base=first_seq, window=window,
                                   keep_first=keep_first, slopes=slopes, temps=temps,
                                   softcap=softcap, pool=pool, k_pool=k_pool, v_pool=v_pool, chunk=chunk)
    if max_q is None:
        max_q = int((cu_q[1:] - cu_q[:-1]).max())
    assert q.stride(2) == 1 and out.is_contiguous() and out.shape == (T, H, E) and out.dtype == q.dtype
    assert k_cache.is_contiguous() and k_cache.dtype == q.dtype
    vs = _value_rows(k_cache, v_cache)
    assert block_tables.dtype == torch.int32 and block_tables.stride(1) == 1
    if gate is not None:
        assert gate.stride(1) == 1 and gate.dtype == q.dtype
    qs_t, qs_h, _ = q.stride()
    # (sizes and strides that the clearing kernel never takes are told without the library's rule, a call of 2 us)
    if clear and (nseq <= 0 or max_q <= 0 or (qs_t | qs_h | D | E | vs) % 8 or _tiles_form(
            q.data_ptr(), qs_t, qs_h, k_cache.data_ptr(), v_cache.data_ptr(), out.data_ptr(), nseq,
            max_q, D, E, vs, _dt(q)) != 2):
        (out[first_seq:] if first_seq else out).zero_()
        clear = False
    _check(_tiles(q.data_ptr(), qs_t, qs_h, k_cache.data_ptr(), v_cache.data_ptr(),
                  block_tables.data_ptr(), block_tables.stride(0), k_cache.shape[1],
                  _i32c(cu_q).data_ptr(), _i32(positions).data_ptr(),
                  _f32(sink).data_ptr() if sink is not None else None,
                  _ptr(gate), gate.stride(0) if gate is not None else 0, out.data_ptr(), scale,
                  nseq, 0, max_q, H, G, D, E, int(window), int(keep_first), _slopes(slopes, H), vs,
                  *_pool_args(k_cache, v_cache, vs, H, temps, softcap, pool, k_pool, v_pool), int(chunk),
                  first_seq if clear else 0, T if clear else 0, _dt(q), _stream()), "sink_attention_prefill")
    return out


def _i32c(t):
    assert t.dtype == torch.int32 and t.stride(0) == 1
    return t


def decode_splits(batch: int, kv_heads: int, heads: int, max_context_len) -> int:
    """Workgroups per (sequence, KV head group) of the split decode kernel: four per CU, each with at least 128
    keys of the longest context; up to eight per CU where one of them would walk more than 2048 keys, for the batch
    that waits for its longest sequence.  64 sequences of 512..1024 keys, 8 KV heads, 2 heads each: 50 us with four,
    54 with eight (float 84 and 88); 64 of 200 keys and one of 8192: 287 and 174 (float 358 and 220)."""
    groups = max(1, batch * kv_heads * -(-(heads // kv_heads) // 4))
    longest = int(max_context_len) if max_context_len else 1024
    want = max(1, 1024 // groups, min(2048 // groups, -(-longest // 2048)))
    return min(16, want, max(1, (longest + 127) // 128))


def next_splits(batch: int, kv_heads: int, heads: int, seen) -> int:
    """Workgroups per (sequence, group of up to 16 heads of a KV head) of the matrix-core decode kernel: one per CU, each
    with at least 512 keys of what a row sees (``seen``); up to eight per CU where one would walk more than 2048 keys, as in
    ``decode_splits``.  The kernel alone in us, 8 KV heads: 4 x 1024 keys 20.7 whole, 8.1 and 4.3 for the fold in four splits;
    1 x 512 11.2 whole, 7.2 and 3.8 in two, which is 19 and 25 a call; 16 x 2048 with 512 workgroups no faster than with 256."""
    groups = max(1, batch * kv_heads * -(-(heads // kv_heads) // 16))
    seen = int(seen) if seen else 1024
    return min(16, max(1, 256 // groups, min(2048 // groups, -(-seen // 2048))), max(1, -(-seen // 512)))


def next_pays(groups: int, R: int, width: int, seen) -> bool:
    """Whether bfloat16 next tokens are the matrix cores': ``groups`` of a sequence and a KV head with ``R`` query heads, keys and
    values of ``width`` together, ``seen`` keys (an upper bound, None if there is none).  A workgroup of theirs takes four waves,
    which walk tiles of 32 keys: 128 keys at a time, and for one or two heads much of the tiles is idle, where the kernel on the
    vector units takes keys one by one.  That shows once the card is full of workgroups, until a context is long.  us, matrix
    cores / vector units:
      one head, 128 + 128 wide: 768 groups of 130 keys 23 / 25, 1024 of 128 19 / 25, of 130 26 / 24, of 260 37 / 33, of 512 56 / 53, of 1030 100 /
      103, 1536 of 200 40 / 34, of 1500 197 / 189, 2560 of 64 32 / 24, of 512 120 / 127, 4096 of 16 49 / 24, of 250 100 / 90, of 256 99 / 93;
      64 + 128: 1024 of 260 32 / 30, of 700 57 / 62, 1536 of 200 34 / 30, of 1030 115 / 104, 8192 of 16 87 / 32
      two heads, 128 + 128: 512 of 260 21 / 24, 1024 of 260 37 / 34, of 512 58 / 56, 2048 of 128 33 / 36, of 512 99 / 104, 4096 of 64 50 / 39, of
      512 189 / 177; four: 1536 of 200 42 / 53, 2048 of 16 30 / 28, of 64 30 / 35
      64 + 64, one head: 1536 of 260 30 / 31, 4096 of 64 25 / 25, 6144 of 16 33 / 25, of 96 38 / 40, 8192 of 64 44 / 40, of 128 56 / 61"""
    if not seen or R > 4:
        return True
    if R > 2:
        return width <= 128 or groups < 2048 or seen > 16
    if width <= 128:
        return groups < 6144 or seen > 64
    return groups * width < (1 << 18 if seen > 128 else 1 << 19) or seen > 1536


def sink_attention_decode(q, k_cache, v_cache, block_tables, context_lens, scale, sink, gate, out,
                          max_context_len=None, window=0, keep_first=0, slopes=None, temps=None,
                          softcap=0.0, pool=0, k_pool=None, v_pool=None, chunk=0, clear=False):
    """Single next tokens: row b is sequence b with ``context_lens[b]`` keys.  bfloat16 rows of 64 / 128 go to the
    matrix cores (``hybrid_next.hip``) where that is faster (``next_pays``), unless pooled rows, temperatures or a soft cap
    belong to the call; those, floats and keys of 256 to the split-context kernel on the vector units; both fold the splits by a second small kernel.  Other sizes go through the row kernel.  ``clear``: ``out`` is new, rows without a
    context become zeros (otherwise they stay as they are)."""
    B, H, D = q.shape
    G, E = k_cache.shape[2], v_cache.shape[3]
    es = q.element_size()
    vs = _value_rows(k_cache, v_cache)
    if (_split_ok(D, E) and q.stride(2) == 1 and q.stride(1) == D and q.data_ptr() % 16 == 0
            and (B == 1 or (q.stride(0) * es) % 16 == 0) and k_cache.is_contiguous()
            and vs % 8 == 0 and v_cache.data_ptr() % 16 == 0 and out.is_contiguous()):
        seen = max_context_len
        if window and seen:           # what a row can see bounds the useful splits
            seen = min(int(seen), int(window) + int(keep_first) + (int(seen) // pool if pool else 0))
        if chunk and seen:
            seen = min(int(seen), int(chunk))
        if q.dtype == torch.bfloat16 and _nxa_ok(D, E) and temps is None and not softcap and not pool \
                and next_pays(B * G, H // G, D + E, seen):
            splits = next_splits(B, G, H, seen)
            ws = torch.empty((B * H * splits * (E + 2),), dtype=torch.float32, device=q.device) if splits > 1 else None
            if gate is not None:
                assert gate.stride(1) == 1 and gate.dtype == q.dtype
            _check(_nxa(q.data_ptr(), q.stride(0) if B > 1 else H * D, D, k_cache.data_ptr(), v_cache.data_ptr(),
                        block_tables.data_ptr(), block_tables.stride(0), k_cache.shape[1], _i32c(context_lens).data_ptr(),
                        None if sink is None else _f32(sink).data_ptr(), _ptr(gate), gate.stride(0) if gate is not None else 0,
                        out.data_ptr(), _ptr(ws), scale, B, H, G, D, E, splits, int(window), int(keep_first),
                        _slopes(slopes, H), vs, int(chunk), int(clear), _stream()), "next_attention")
            return out
        splits = decode_splits(B, G, H, seen)
        ws = torch.empty((B * H * splits * (E + 2),), dtype=torch.float32, device=q.device)
        if gate is not None:
            assert gate.stride(1) == 1 and gate.dtype == q.dtype
        _check(_split(q.data_ptr(), q.stride(0) if B > 1 else H * D, q.stride(1), k_cache.data_ptr(),
                      v_cache.data_ptr(), block_tables.data_ptr(), block_tables.stride(0),
                      k_cache.shape[1], _i32c(context_lens).data_ptr(),
                      _f32(sink).data_ptr() if sink is not None else None,
                      _ptr(gate), gate.stride(0) if gate is not None else 0, out.data_ptr(),
                      ws.data_ptr(), scale, B, H, G, D, E, splits, int(window), int(keep_first),
                      _slopes(slopes, H), vs,
                      *_pool_args(k_cache, v_cache, vs, H, temps, softcap, pool, k_pool, v_pool), int(chunk),
                      int(clear), _dt(q), _stream()),
               "sink_attention_decode")
        return out
    if clear:
        out.zero_()
    return _attention_rows(q, k_cache, v_cache, block_tables, None, context_lens, 0, scale, sink,
                           gate, out, 0, window, keep_first, slopes, temps, softcap, pool, k_pool, v_pool,
                           chunk)


def _rows_out(T, H, E, slots, device):
    """The output rows of a recurrence: its kernel clears those that no sequence owns itself."""
    new = torch.empty if slots.shape[0] else torch.zeros
    return new((T, H, E), dtype=torch.float32, device=device)


# ------------------------------------------------------------------ gated delta rule
def delta_prepare(q, k, v, b, a, conv_w, a_log, dt_bias, conv_state, cu_q, positions, slots,
                  row_seq, conv_bias=None, ssd=False):
    T, G, D = q.shape
    H, E = v.shape[1], v.shape[2]
    rs = q.stride(0)
    base = q.data_ptr()
    es = q.element_size()
    # q, k, v are the first three column blocks of one projection output, b a view of it; a is a
    # view of it too or a tensor of its own, [T, H] (a decay per head) or [T, H*D] (per key channel)
    assert k.data_ptr() == base + G * D * es and v.data_ptr() == base + 2 * G * D * es
    assert T == 1 or (k.stride(0) == rs and v.stride(0) == rs and (ssd or b.stride(0) == rs))
    assert a.dtype == q.dtype and a.stride(-1) == 1 and a.shape[-1] in (H, H * D)
    DC = a.shape[-1] // H
    assert dt_bias.numel() == H * DC and (not ssd or DC == 1)
    b_off = 0 if ssd else (b.data_ptr() - base) // es
    if conv_bias is not None:
        assert conv_bias.numel() == 2 * G * D + H * E
    dev = q.device
    taps = _f32(conv_w).shape[1]
    assert conv_w.shape[0] == 2 * G * D + H * E
    f = dict(dtype=torch.float32, device=dev)
    qn, kn = torch.empty((T, G, D), **f), torch.empty((T, G, D), **f)
    vv, beta = torch.empty((T, H, E), **f), torch.empty((T, H), **f)
    decay = torch.empty((T, H) if DC == 1 else (T, H, D), **f)
    if cu_q is not None:
        assert row_seq is not None, "prefill-form steps pass the sequence of each row"
    B = slots.shape[0]
    _check(_prep(base, rs if T > 1 else int(rs or 0), b_off, a.data_ptr(), a.stride(0), DC,
                 conv_w.data_ptr(), taps, _ptr(_f32(conv_bias)) if conv_bias is not None else None,
                 int(bool(ssd)), _f32(a_log).data_ptr(), _f32(dt_bias).data_ptr(), _f32(conv_state).data_ptr(), _ptr(_i32(cu_q)),
                 _i32(positions).data_ptr(), _i32(slots).data_ptr(),
                 _ptr(_i32(row_seq)) if cu_q is not None else None, qn.data_ptr(), kn.data_ptr(),
                 vv.data_ptr(), beta.data_ptr(), decay.data_ptr(), T, B, H, G, D, E, _dt(q),
                 _stream()), "delta_prepare")
    return qn, kn, vv, beta, decay


def delta_scan(qn, kn, vv, beta, decay, state, cu_q, positions, slots, correct=True):
    T, G, D = qn.shape
    H, E = vv.shape[1], vv.shape[2]
    assert state.shape[1:] == (H, D, E)
    o = _rows_out(T, H, E, slots, qn.device)
    if decay.dim() == 3:                 # a decay per head and key channel
        assert decay.shape == (T, H, D) and decay.is_contiguous() and correct
        _check(_cscan(qn.data_ptr(), kn.data_ptr(), vv.data_ptr(), beta.data_ptr(), decay.data_ptr(),
                      _f32(state).data_ptr(), _ptr(_i32(cu_q)), _i32(positions).data_ptr(),
                      _i32(slots).data_ptr(), o.data_ptr(), T, slots.shape[0], H, G, D, E, _stream()),
               "channel_delta_scan")
        return o
    # prompt portions in chunks on the matrix cores need a place for what a first kernel works out
    ws = None
    if cu_q is not None:
        n = _scan_ws(qn.data_ptr(), kn.data_ptr(), vv.data_ptr(), cu_q.data_ptr(), o.data_ptr(), T,
                     slots.shape[0], H, G, D, E)
        ws = torch.empty((n,), dtype=torch.uint8, device=qn.device) if n else None
    _check(_scan(qn.data_ptr(), kn.data_ptr(), vv.data_ptr(), beta.data_ptr(), decay.data_ptr(),
                 _f32(state).data_ptr(), _ptr(_i32(cu_q)), _i32(positions).data_ptr(),
                 _i32(slots).data_ptr(), o.data_ptr(), _ptr(ws), T, slots.shape[0], H, G, D, E, int(bool(correct)),
                 _stream()), "delta_scan")
    return o


@functools.lru_cache(maxsize=64)
def _delta_next_sizes(H, G, D, E, taps) -> bool:
    return bool(_next_ok(H, G, D, E, taps))


def delta_next_pays(B: int, H: int, D: int, E: int) -> bool:
    """Whether single next tokens of ``B`` sequences are fewer than the three calls pay for.  From 256 MB of state the card's
    time is the state's alone, and the step's own kernel, with smaller workgroups, moves it faster; heads of small states
    are bound by their workgroups.  One kernel / three, us, bfloat16: 16 / 8 heads of 128 x 128 64 sequences 32 / 55, 192 78 /
    84, 256 116 / 109; 32 / 8 of them 96 81 / 82, 128 122 / 110; 16 / 8 of 64 x 64 256 44 / 53, 512 78 / 64."""
    return B * H * D * E < 1 << 26 and B * H <= 4096


def delta_next(proj, a, gate, sizes, conv_w, a_log, dt_bias, norm_w, conv_state, state, positions, slots, eps, out_dtype, act):
    """Single next tokens: ``delta_prepare``, ``delta_scan`` and ``gated_head_norm`` in one kernel, their sums in the same order; None where
    it has no instance or they are too many (``delta_next_pays``; the caller then makes the three calls).  ``proj`` [T, ..] = [q | k | v | gate | beta | decay | ..]
    with ``a`` and ``gate`` None, or [q | k | v | beta | ..] with ``a`` [T, H*D] (a decay per key channel) and ``gate`` [T, H*E]."""
    H, G, D, E = sizes
    T, C, taps = proj.shape[0], 2 * G * D + H * E, conv_w.shape[1]
    if not (T > 0 and slots.shape[0] == T and proj.dtype == out_dtype and out_dtype in _DT and delta_next_pays(T, H, D, E)
            and _delta_next_sizes(H, G, D, E, taps) and proj.stride(1) == 1 and conv_w.shape[0] == C and state.data_ptr() % 16 == 0):
        return None
    base, row, es = proj.data_ptr(), proj.stride(0), proj.element_size()
    if a is None:
        assert gate is None and proj.shape[1] >= C + H * E + 2 * H
        DC, b_off, ap, a_row, gp, gate_row = 1, C + H * E, base + (C + H * E + H) * es, row, base + C * es, row
    else:
        if a.dtype != out_dtype or gate.dtype != out_dtype or a.shape != (T, H * D) or gate.shape != (T, H * E) \
                or a.stride(1) != 1 or gate.stride(1) != 1 or proj.shape[1] < C + H:
            return None
        DC, b_off, ap, a_row, gp, gate_row = D, C, a.data_ptr(), a.stride(0), gate.data_ptr(), gate.stride(0)
    assert state.shape[1:] == (H, D, E) and dt_bias.numel() == H * DC and norm_w.numel() in (E, H * E)
    assert act in ("silu", "sigmoid")
    out = torch.empty((T, H * E), dtype=out_dtype, device=proj.device)
    _check(_next(base, row, b_off, ap, a_row, DC, gp, gate_row, _f32(conv_w).data_ptr(), taps, _f32(a_log).data_ptr(),
                 _f32(dt_bias).data_ptr(), _f32(norm_w).data_ptr(), norm_w.numel() == H * E and H > 1,
                 _f32(conv_state).data_ptr(), _f32(state).data_ptr(), _i32(positions).data_ptr(), _i32(slots).data_ptr(),
                 out.data_ptr(), eps, act == "sigmoid", T, H, G, D, E, _DT[out_dtype], _stream()), "delta_next")
    return out


def delta_scan_workspace(tokens: int, seqs: int, H: int, G: int, D: int, E: int) -> int:
    """The most bytes ``delta_scan`` takes for itself in a step of up to that many tokens and sequences: it grows with
    both, and steps of too few tokens for their sequences take none."""
    seqs = min(seqs, tokens, max(tokens // 20, tokens - 1024))
    aligned = 256
    return _scan_ws(aligned, aligned, aligned, aligned, aligned, tokens, seqs, H, G, D, E) if seqs > 0 else 0


def gated_head_norm(o, w, gate, eps, out_dtype, act="silu"):
    T, H, E = o.shape
    assert gate.stride(-1) == 1 and gate.dtype == out_dtype and w.numel() in (E, H * E)
    assert act in ("silu", "sigmoid")
    out = torch.empty((T, H, E), dtype=out_dtype, device=o.device)
    _check(_ghn(_f32(o).data_ptr(), _f32(w).data_ptr(), gate.data_ptr(), gate.stride(0),
                out.data_ptr(), T, H, E, eps, int(w.numel() == H * E and H > 1), int(act == "sigmoid"),
                _dt(out), _stream()), "gated_head_norm")
    return out


# ------------------------------------------------------------------ grouped expert routing
def grouped_route(h, router_w, top, groups, keep, score="softmax", bias=None, gates=0):
    T, W = h.shape
    if score == "chosen":
        NR = router_w.shape[0]
        assert groups == 1 and keep == 1 and h.is_contiguous() and 0 <= gates < NR
        dense = torch.empty((T, NR), dtype=torch.float32, device=h.device)
        _check(_crt(h.data_ptr(), _f32(router_w).data_ptr(), _ptr(_f32(bias)) if bias is not None else None,
                    dense.data_ptr(), T, W, NR - gates, NR, top, _dt(h), _stream()), "chosen_route")
        return dense
    assert score in ("softmax", "sigmoid") and bias is None and not gates
    NE = router_w.shape[0]
    assert h.is_contiguous()
    dense = torch.empty((T, NE), dtype=torch.float32, device=h.device)
    _check(_route(h.data_ptr(), _f32(router_w).data_ptr(), dense.data_ptr(), T, W, NE, top, groups,
                  keep, int(score == "sigmoid"), _dt(h), _stream()), "grouped_route")
    return dense


def gelu_route_scale(up, dense, ff, out_dtype):
    T = up.shape[0]
    NE = dense.shape[1]
    assert up.is_contiguous() and up.dtype == out_dtype and up.shape[1] == NE * ff
    act = torch.empty_like(up)
    _check(_gelu(up.data_ptr(), _f32(dense).data_ptr(), act.data_ptr(), T, NE, ff, _dt(up),
                 _stream()), "gelu_route_scale")
    return act


def swiglu_route_scale(gu, dense, ff, shared_ff, out_dtype):
    T = gu.shape[0]
    C = gu.shape[1] // 2
    NE = dense.shape[1] if dense is not None else 0
    assert gu.stride(1) == 1 and gu.dtype == out_dtype and C == NE * ff + shared_ff
    act = torch.empty((T, C), dtype=out_dtype, device=gu.device)
    _check(_swi(gu.data_ptr(), _rows(gu), _ptr(_f32(dense)) if dense is not None else None,
                act.data_ptr(), T, NE, ff if NE else 1, shared_ff, _dt(gu), _stream()),
           "swiglu_route_scale")
    return act


# ------------------------------------------------------------------ positions, grouped norms
def embed_sinusoid(ids, positions, table, inv_freq):
    T, W = ids.shape[0], table.shape[1]
    assert table.is_contiguous() and inv_freq.numel() == W // 2
    x = torch.empty((T, W), dtype=torch.float32, device=table.device)
    _check(_esin(_i32(ids).data_ptr(), _i32(positions).data_ptr(), table.data_ptr(),
                 _f32(inv_freq).data_ptr(), x.data_ptr(), T, W, _dt(table), _stream()), "embed_sinusoid")
    return x


def group_rms_norm(x, w, groups, eps, out_dtype):
    return residual_group_norm(x, (), w, groups, eps, out_dtype)


def residual_group_norm(x, ys, w_next, groups, eps, out_dtype):
    x = _f32(x)
    T, W = x.shape
    ys = list(ys)
    assert len(ys) <= 2, "at most two branches are added per call"
    for y in ys:
        assert y.shape == x.shape and y.stride(1) == 1 and y.dtype == out_dtype
    h = torch.empty((T, W), dtype=out_dtype, device=x.device) if w_next is not None else None
    if h is None and not ys:
        return None
    y1 = ys[0] if ys else None
    y2 = ys[1] if len(ys) > 1 else None
    _check(_rgn(x.data_ptr(), _ptr(y1), _rows(y1) if y1 is not None else 0, _ptr(y2),
                _rows(y2) if y2 is not None else 0, _ptr(w_next), _ptr(h), T, W, groups, eps,
                _DT[out_dtype], _stream()), "residual_group_norm")
    return h


def add_normed_mean(x, parts, eps):
    x = _f32(x)
    T, W = x.shape
    assert 1 <= len(parts) <= 2
    (y1, w1), (y2, w2) = parts[0], (parts[1] if len(parts) > 1 else (None, None))
    for y in (y1, y2):
        assert y is None or (y.shape == x.shape and y.stride(1) == 1 and y.dtype == y1.dtype)
    _check(_anm(x.data_ptr(), y1.data_ptr(), _rows(y1), _f32(w1).data_ptr(), _ptr(y2),
                _rows(y2) if y2 is not None else 0, _f32(w2).data_ptr() if w2 is not None else None,
                T, W, eps, _dt(y1), _stream()), "add_normed_mean")


def unit_norm_store(q, k, eps, k_cache, v_cache, slot_mapping):
    T, H, D = q.shape
    G = k.shape[1]
    rs = q.stride(0)
    assert (T == 1 or k.stride(0) == rs) and q.stride(1) == D and k.stride(1) == D \
        and q.stride(2) == 1 and k.stride(2) == 1, "q / k must be views of one projection output"
    if k_cache is not None:
        assert k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.dtype == q.dtype \
            and k_cache.shape[2:] == (G, D) and v_cache.shape[2:] == (G, D)
    _check(_uns(q.data_ptr(), k.data_ptr(), rs, eps, _ptr(k_cache), _ptr(v_cache),
                _ptr(_i32(slot_mapping)), T, H, G, D, _dt(q), _stream()), "unit_norm_store")


def tanh_cap_(z, cap):
    assert z.is_contiguous()
    _check(_cap(z.data_ptr(), z.numel(), cap, _dt(z), _stream()), "tanh_cap")
    return z


# ------------------------------------------------------------------ gated outer-product recurrences
def _heads_view(t, n):
    """Element stride per token of a [T, heads, n] view whose heads are dense."""
    assert t.stride(2) == 1 and t.stride(1) == n
    return _rows(t)


def mlstm_scan(q, k, v, i_raw, f_raw, i_bias, f_bias, cap, state, norm_state, max_state,
               cu_q, positions, slots, longest=0):
    T, H, D = q.shape
    E = v.shape[2]
    ZG = (E + 15) // 16
    assert state.shape[1:] == (H, D, E) and norm_state.shape[1:] == (H, ZG, D) \
        and max_state.shape[1:] == (H, ZG)
    assert i_raw.shape == (T, H) and f_raw.shape == (T, H) and i_raw.stride(1) == 1 and f_raw.stride(1) == 1
    assert T == 1 or i_raw.stride(0) == f_raw.stride(0)
    assert k.dtype == q.dtype and v.dtype == q.dtype and i_raw.dtype == q.dtype and f_raw.dtype == q.dtype
    o = _rows_out(T, H, E, slots, q.device)
    rows, ws = (q.data_ptr(), k.data_ptr(), v.data_ptr(), _heads_view(q, D), _heads_view(k, D), _heads_view(v, E)), None
    if cu_q is not None:
        n = _mlstm_bytes(*rows, T, slots.shape[0], int(longest or 0), H, D, E, _dt(q))
        if n:
            ws = torch.empty((n,), dtype=torch.uint8, device=q.device)
    _check(_mlstm(*rows, i_raw.data_ptr(), f_raw.data_ptr(), _rows(i_raw),
                  _f32(i_bias).data_ptr(), _f32(f_bias).data_ptr(), cap, _f32(state).data_ptr(),
                  _f32(norm_state).data_ptr(), _f32(max_state).data_ptr(), _ptr(_i32(cu_q)),
                  _i32(positions).data_ptr(), _i32(slots).data_ptr(), o.data_ptr(), _ptr(ws), T,
                  slots.shape[0], H, D, E, _dt(q), _stream()), "mlstm_scan")
    return o


def mlstm_norm(proj, sizes, i_bias, f_bias, cap, norm_w, state, norm_state, max_state, cu_q, positions, slots, eps, out_dtype,
               longest=0):
    """``mlstm_scan`` and ``gated_head_norm`` (sigmoid) in one call: ``proj`` [T, ..] = [q | k | v | gate | input gate | forget
    gate] -> [T, H*E].  None where the two calls are to be made.  (8 next tokens: a layer's call 35 us as two, 22 as one.)"""
    H, D, E = sizes
    T, B, HD, HE, dt = proj.shape[0], slots.shape[0], H * D, H * E, _DT.get(out_dtype)
    if dt is None or proj.dtype != out_dtype or proj.stride(1) != 1 or not T or not B or proj.shape[1] != 2 * (HD + HE + H):
        return None
    ZG = (E + 15) // 16
    assert state.shape[1:] == (H, D, E) and norm_state.shape[1:] == (H, ZG, D) and max_state.shape[1:] == (H, ZG)
    assert norm_w.numel() in (E, HE)
    base, row, es, n = proj.data_ptr(), _rows(proj), 2 if dt == 0 else 4, 0
    if cu_q is not None:
        n = _mlstm_bytes(base, base + HD * es, base + 2 * HD * es, row, row, row, T, B, int(longest or 0), H, D, E, dt)
    out = -(-T * HE * 4 // 256) * 256
    ws = torch.empty((out + n,), dtype=torch.uint8, device=proj.device)
    y = torch.empty((T, HE), dtype=out_dtype, device=proj.device)
    o = ws.data_ptr()
    _check(_mlstm_rows(base, row, _f32(i_bias).data_ptr(), _f32(f_bias).data_ptr(), cap, _f32(state).data_ptr(),
                       _f32(norm_state).data_ptr(), _f32(max_state).data_ptr(), _ptr(_i32(cu_q)), _i32(positions).data_ptr(),
                       _i32(slots).data_ptr(), o, o + out if n else None, y.data_ptr(), _f32(norm_w).data_ptr(),
                       norm_w.numel() == HE and H > 1, eps, T, B, H, D, E, dt, _stream()), "mlstm_norm")
    return y


def mlstm_scan_workspace(tokens: int, seqs: int, H: int, D: int, E: int) -> int:
    """The most bytes ``mlstm_scan`` takes for itself in a step of up to that many tokens and sequences."""
    seqs = min(seqs, tokens)
    return (tokens // 64 + seqs) * H * 1024 if seqs > 0 else 0


_channel_bytes = functools.lru_cache(maxsize=256)(_chan_bytes)


def _channel_chunks(rule, q, k, v, a_raw, a_bias, bonus, tau, qscale, state, cu_q, positions, slots,
                    longest):
    """Prompt portions in chunks side by side, None where the rows are to be walked token by token.  (The callers look at the
    portions' lengths first, as the library's rule does: most steps that it turns down do not come here, 1.2 us of a call.)"""
    T, H, D = q.shape
    E, B = v.shape[2], slots.shape[0]
    dt, v_row = _dt(q), _rows(v)
    n = _channel_bytes(T, B, longest, H, D, E, v.data_ptr() % 16 == 0 and v_row % (8 if dt == 0 else 4) == 0, False, dt)
    if not n:
        return None
    o = torch.empty((T, H, E), dtype=torch.float32, device=q.device)
    ws = torch.empty((n,), dtype=torch.uint8, device=q.device)
    _check(_chan(rule, q.data_ptr(), k.data_ptr(), v.data_ptr(), _heads_view(q, D), _heads_view(k, D), _heads_view(v, E),
                 a_raw.data_ptr(), _rows(a_raw), _f32(a_bias).data_ptr(), _ptr(bonus), tau, qscale, _f32(state).data_ptr(),
                 _i32(cu_q).data_ptr(), _i32(positions).data_ptr(), _i32(slots).data_ptr(), ws.data_ptr(), o.data_ptr(), None,
                 None, 0, None, 0, 0.0, 0, T, B, H, D, E, dt, _stream()), "channel_chunks")
    return o


def channel_scan_workspace(tokens: int, seqs: int, H: int, D: int, E: int) -> int:
    """Bytes that ``gla_scan`` / ``wkv_scan`` take at most for themselves in a step of up to that many tokens and sequences:
    they grow with both, and steps of too few tokens for their sequences take none."""
    seqs = min(seqs, max(tokens // 64, (2 * tokens - 126) // 3))
    return _channel_bytes(tokens, seqs, -1, H, D, E, True, True, 0) if seqs > 0 else 0


def _check_gla(q, k, v, a_raw, a_bias, state):
    T, H, D = q.shape
    assert state.shape[1:] == (H, D, v.shape[2]) and a_raw.shape == (T, H * D) and a_raw.stride(1) == 1
    assert k.dtype == q.dtype and v.dtype == q.dtype and a_raw.dtype == q.dtype
    assert a_bias.numel() == H * D


def gla_scan(q, k, v, a_raw, a_bias, tau, state, cu_q, positions, slots, longest=0):
    T, H, D = q.shape
    E, B = v.shape[2], slots.shape[0]
    _check_gla(q, k, v, a_raw, a_bias, state)
    if cu_q is not None and (T >= 96 * B or 2 * (longest or 0) >= 192 + B):
        o = _channel_chunks(0, q, k, v, a_raw, a_bias, None, tau, D ** -0.5, state, cu_q, positions, slots,
                            int(longest or 0))
        if o is not None:
            return o
    o = _rows_out(T, H, E, slots, q.device)
    _check(_gla(q.data_ptr(), k.data_ptr(), v.data_ptr(), _heads_view(q, D), _heads_view(k, D),
                _heads_view(v, E), a_raw.data_ptr(), _rows(a_raw), _f32(a_bias).data_ptr(), tau,
                _f32(state).data_ptr(), _ptr(_i32(cu_q)), _i32(positions).data_ptr(),
                _i32(slots).data_ptr(), o.data_ptr(), T, B, H, D, E, _dt(q), _stream()),
           "gla_scan")
    return o


def gla_norm(proj, a_raw, sizes, a_bias, tau, norm_w, state, cu_q, positions, slots, eps, out_dtype, longest=0):
    """``gla_scan`` and ``gated_head_norm`` (silu) in one call: ``proj`` [T, ..] = [q | k | v | gate | ..] -> [T, H*E]; prompt
    portions in chunks are normed where they are formed.  None where the two calls are to be made.  (64 next tokens: a layer's
    call 34 us as two, 22 as one, most of it the calls themselves.)"""
    H, D, E = sizes
    T, B, HD, HE, dt = proj.shape[0], slots.shape[0], H * D, H * E, _DT.get(out_dtype)
    if dt is None or proj.dtype != out_dtype or a_raw.dtype != out_dtype or proj.stride(1) != 1 or not T or not B \
            or a_raw.shape != (T, HD) or a_raw.stride(1) != 1 or proj.shape[1] < 2 * (HD + HE):
        return None
    base, row, es, n = proj.data_ptr(), _rows(proj), 2 if dt == 0 else 4, 0
    v, gate, wp = base + 2 * HD * es, base + (2 * HD + HE) * es, _f32(norm_w).data_ptr()
    if cu_q is not None and (T >= 64 * B or 2 * (longest or 0) >= 128 + B):      # (of the library's rule)
        n = _channel_bytes(T, B, int(longest or 0), H, D, E, (v | gate | wp) % 16 == 0 and row % (8 if dt == 0 else 4) == 0,
                           True, dt)
    assert state.shape[1:] == (H, D, E) and a_bias.numel() == HD and norm_w.numel() in (E, HE)
    y = torch.empty((T, HE), dtype=out_dtype, device=proj.device)
    if not n:
        o = torch.empty((T, H, E), dtype=torch.float32, device=proj.device)
        _check(_gla_rows(base, row, a_raw.data_ptr(), _rows(a_raw), _f32(a_bias).data_ptr(), tau, _f32(state).data_ptr(),
                         _ptr(_i32(cu_q)), _i32(positions).data_ptr(), _i32(slots).data_ptr(), o.data_ptr(), y.data_ptr(), wp,
                         norm_w.numel() == HE and H > 1, eps, T, B, H, D, E, dt, _stream()), "gla_norm")
        return y
    ws = torch.empty((n,), dtype=torch.uint8, device=proj.device)
    _check(_chan(0, base, base + HD * es, v, row, row, row, a_raw.data_ptr(), a_raw.stride(0), _f32(a_bias).data_ptr(), None,
                 tau, D ** -0.5, _f32(state).data_ptr(), _i32(cu_q).data_ptr(), _i32(positions).data_ptr(),
                 _i32(slots).data_ptr(), ws.data_ptr(), None, y.data_ptr(), gate, row, wp, norm_w.numel() == HE and H > 1,
                 eps, 0, T, B, H, D, E, dt, _stream()), "gla_norm")
    return y


# ------------------------------------------------------------------ scaled branches, latent keys
def rms_norm_rows(x, w, eps, out_dtype):
    T, n = x.shape
    assert x.stride(1) == 1 and x.dtype == out_dtype and w.numel() == n
    out = torch.empty((T, n), dtype=out_dtype, device=x.device)
    _check(_rnr(x.data_ptr(), _rows(x), _f32(w).data_ptr(), out.data_ptr(), T, n, eps, _dt(x),
                _stream()), "rms_norm_rows")
    return out


def residual_sum_norm(x, ys, scales, gain, eps, out_dtype):
    x = _f32(x)
    T, W = x.shape
    ys = list(ys)
    assert len(ys) <= 4 and len(ys) == len(scales), "at most four branches are added per call"
    for y in ys:
        assert y.shape == x.shape and y.stride(1) == 1 and y.dtype == out_dtype
    h = torch.empty((T, W), dtype=out_dtype, device=x.device) if gain is not None else None
    if h is None and not ys:
        return None
    n = len(ys)
    ptrs = (ctypes.c_void_p * 4)(*[y.data_ptr() for y in ys], *([None] * (4 - n)))
    strides = (ctypes.c_long * 4)(*[_rows(y) for y in ys], *([0] * (4 - n)))
    sc = (ctypes.c_float * 4)(*[float(v) for v in scales], *([0.0] * (4 - n)))
    _check(_rsn(x.data_ptr(), *map(ctypes.addressof, (ptrs, strides, sc)), n, float(gain) if gain is not None else 0.0,
                _ptr(h), T, W, eps, _DT[out_dtype], _stream()), "residual_sum_norm")
    return h


def row_norm_store(q, k, v, qw, kw, eps, k_cache, v_cache, slot_mapping):
    T, H, D = q.shape
    G, E = v.shape[1], v.shape[2]
    rs = q.stride(0)
    assert (T == 1 or (k.stride(0) == rs and v.stride(0) == rs)) and q.stride(1) == D \
        and k.stride(1) == D and v.stride(1) == E and q.stride(2) == 1 and k.stride(2) == 1 \
        and v.stride(2) == 1, "q / k / v must be views of one projection output"
    assert (qw is None) == (kw is None)
    if qw is not None:
        assert qw.numel() == H * D and kw.numel() == G * D
    if k_cache is not None:
        assert k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.dtype == q.dtype \
            and k_cache.shape[2:] == (G, D) and v_cache.shape[2:] == (G, E)
    _check(_rns(q.data_ptr(), k.data_ptr(), v.data_ptr(), rs, _ptr(_f32(qw)) if qw is not None else None,
                _ptr(_f32(kw)) if kw is not None else None, eps, _ptr(k_cache), _ptr(v_cache),
                _ptr(_i32(slot_mapping)), T, H * D, G * D, G * E, _dt(q), _stream()), "row_norm_store")


def latent_rope_store(q_abs, q, dkv, w, eps, positions, inv_freq, rot_dims, k_cache, v_cache,
                      slot_mapping, neighbours=False, mult=1.0, assemble=True):
    T, H, R = q.shape[0], q.shape[1], w.numel()
    P = dkv.shape[1] - R
    D = q.shape[2] - P
    assert dkv.dtype == q.dtype and (q_abs is not None or not assemble)
    assert q_abs is None or (q_abs.is_contiguous() and q_abs.dtype == q.dtype and q_abs.shape == (H, T, R))
    assert q.shape[:2] == (T, H) and q.stride(2) == 1 and q.stride(1) == D + P and dkv.stride(1) == 1
    assert w.numel() == R and inv_freq.numel() * 2 == rot_dims
    if k_cache is not None:
        assert k_cache.is_contiguous() and k_cache.dtype == q.dtype and k_cache.shape[2:] == (1, R + P)
        if v_cache is not None:          # None: the values are the leading part of the key rows
            assert v_cache.is_contiguous() and v_cache.shape[2:] == (1, R)
    out = torch.empty((T, H, R + P if assemble else P), dtype=q.dtype, device=q.device)
    _check(_lrs(q_abs.data_ptr() if assemble else None, q.data_ptr(), _rows(q), dkv.data_ptr(), _rows(dkv),
                _f32(w).data_ptr(), eps, _i32(positions).data_ptr(), _f32(inv_freq).data_ptr(),
                int(rot_dims), _ptr(k_cache), _ptr(v_cache), _ptr(_i32(slot_mapping)), out.data_ptr(),
                T, H, D, P, R, int(neighbours), float(mult), _dt(q), _stream()), "latent_rope_store")
    return out


# ------------------------------------------------------------------ attention over shared latents
def latent_attention_ok(q_abs, k_cache, rot_dim: int) -> bool:
    """True when the matrix-core kernel has an instance: bfloat16, latents of up to 512 numbers,
    sizes in whole runs of eight."""
    return bool(q_abs.dtype == torch.bfloat16 and k_cache is not None and k_cache.dtype == torch.bfloat16
                and k_cache.is_contiguous() and rot_dim > 0 and _lat_ok(q_abs.shape[2], rot_dim))


def latent_splits(batch: int, heads: int, latent: int, max_context_len, window: int = 0) -> int:
    """Workgroups per sequence and 32 query rows for single next tokens: one per compute unit for
    latents above 256 numbers (a workgroup fills its LDS and registers), several below, each with at
    least 128 keys of the longest context."""
    tiles = batch * -(-heads // 32) if heads <= 64 else batch * -(-heads // 128)
    want = -(-(256 if latent > 256 else 768) // max(tiles, 1))
    seen = min(int(max_context_len), window + 31) if window and max_context_len else max_context_len
    room = max(1, (int(seen) + 127) // 128) if seen else 8
    return max(1, min(16, want, room))


def _latent(q_abs, q_rot, k_cache, tables, cu_q, positions, lens, scale, sink, out, nseq, max_q, window, splits):
    H, T, R = q_abs.shape
    P = q_rot.shape[2]
    assert q_abs.stride(2) == 1 and q_rot.stride(2) == 1 and q_rot.shape[:2] == (T, H)
    assert out.shape == (T, H, R) and out.stride(2) == 1 and k_cache.is_contiguous() \
        and k_cache.shape[2:] == (1, R + P) and q_abs.dtype == q_rot.dtype == out.dtype == k_cache.dtype
    assert tables.dtype == torch.int32 and tables.stride(1) == 1 and tables.shape[0] >= nseq
    ws = None
    if splits > 1:
        assert out.is_contiguous()
        ws = torch.empty((nseq * H * splits * (R + 2),), dtype=torch.float32, device=out.device)
    _check(_lat(q_abs.data_ptr(), q_abs.stride(1), q_abs.stride(0), q_rot.data_ptr(), q_rot.stride(0),
                q_rot.stride(1), k_cache.data_ptr(), tables.data_ptr(), tables.stride(0), k_cache.shape[1],
                _ptr(cu_q), _ptr(positions), _ptr(lens), _ptr(_f32(sink)) if sink is not None else None,
                out.data_ptr(), out.stride(0), out.stride(1), _ptr(ws), float(scale), nseq, int(max_q), H, R,
                P, int(window), int(splits), _stream()), "latent_attention")
    return out


def latent_attention_prefill(q_abs, q_rot, k_cache, cu_q, block_tables, positions, scale, sink, out,
                             max_q, window=0):
    """Prompt portions: ``q_abs`` [H, T, R] and ``q_rot`` [T, H, P] are the two parts of the queries,
    sequence b owns rows cu_q[b] .. cu_q[b+1] (absolute rows) and block table row b; ``max_q``: the
    longest portion (a host integer)."""
    nseq = cu_q.shape[0] - 1
    if max_q is None:
        max_q = int((cu_q[1:] - cu_q[:-1]).max())
    return _latent(q_abs, q_rot, k_cache, block_tables, _i32c(cu_q), _i32(positions), None, scale, sink, out,
                   nseq, max_q, window, 1)


def latent_attention_decode(q_abs, q_rot, k_cache, block_tables, context_lens, scale, sink, out,
                            max_context_len=None, window=0):
    """Single next tokens: row b is sequence b with ``context_lens[b]`` keys."""
    B, H, R = out.shape
    return _latent(q_abs, q_rot, k_cache, block_tables, None, None, _i32c(context_lens), scale, sink, out,
                   B, 1, window, latent_splits(B, H, R, max_context_len, window))


# Up to where few rows pay against the library's two products and the calls around them, which take 80 to 90 us
# until the card is full: by the rows of the caches and of the weights that a workgroup walks (rows times rank), and by the
# products (rows times rank times heads; single next tokens are split over their contexts, with sums to be joined, and
# fill the card sooner).  This / those, us:
#   16 heads: R 512 8 portions of 64 53 / 88, of 128 82 / 83, one of 200 58 / 84, of 500 108 / 105; R 256 8 of 128 50 / 84,
#   one of 1000 124 / 125, of 2000 225 / 208; R 128 one of 1000 71 / 84, of 2000 119 / 120
#   64 heads: R 512 8 portions of 16 53 / 87, one of 200 109 / 89, 64 of 8 130 / 82; R 256 2 of 128 53 / 90, 8 of 128 109 / 83;
#   R 128 64 of 8 39 / 80, one of 1000 114 / 102; 128 heads, R 512: one of 64 67 / 87, 8 of 16 96 / 85
#   single next tokens, 512 keys each: 16 heads, R 512 one 29 / 79, 64 45 / 83, 256 56 / 80; 128 heads, R 512 32 84 / 88, 64
#   135 / 101, R 256 64 69 / 90, 128 101 / 99; 64 heads, R 512 64 79 / 89, 256 134 / 104
LATENT_ROWS = 1 << 18


def latent_rows_pay(T: int, H: int, R: int, prompts: bool) -> bool:
    """Whether ``T`` rows are few enough for ``latent_rows``."""
    return T * R <= LATENT_ROWS and T * R * H <= (5 << 20 if prompts else 3 << 20)


def latent_rows(q, dkv, norm_w, eps, positions, inv_freq, rot_dims, neighbours, mult, k_cache, slot_mapping, up_k, up_v,
                block_tables, cu_q, lens, scale, sink, max_q, max_context_len, window=0):
    """A step of few rows from its projections to [T, H, E], in the latents' coordinates, in one call: prompt portions
    (``cu_q``, ``max_q``) or single next tokens (``lens``).  None where the calls are to be made one by one: beyond
    ``latent_rows_pay``, other types than bfloat16, sizes or addresses that are no whole runs of eight."""
    T, H, width = q.shape
    _, D, R = up_k.shape
    E, P = up_v.shape[2], width - D
    if not latent_rows_pay(T, H, R, cu_q is not None) or T == 0 or q.dtype != torch.bfloat16 or not _latr_ok(H, D, P, R, E, int(rot_dims), int(neighbours)):
        return None
    if k_cache is None or any(t.dtype != torch.bfloat16 for t in (dkv, up_k, up_v, k_cache)) or dkv.shape[1] != R + P \
            or slot_mapping is None or block_tables is None:
        return None
    q_row, dkv_row = (q.stride(0), dkv.stride(0)) if T > 1 else (0, 0)
    qp, dp, cp, kp, vp, wp = (t.data_ptr() for t in (q, dkv, k_cache, up_k, up_v, norm_w))
    if (qp | dp | cp | kp | vp | wp) % 16 or (q_row | dkv_row) % 8 or q.stride(2) != 1 or q.stride(1) != width \
            or dkv.stride(1) != 1 or not (up_k.is_contiguous() and up_v.is_contiguous() and k_cache.is_contiguous()):
        return None
    assert k_cache.shape[2:] == (1, R + P) and norm_w.numel() == R and inv_freq.numel() * 2 == rot_dims
    assert block_tables.dtype == torch.int32 and block_tables.stride(1) == 1
    if cu_q is None:
        nseq, max_q, splits = T, 1, latent_splits(T, H, R, max_context_len, window)
        assert lens.shape[0] == T
    else:
        nseq, splits = cu_q.shape[0] - 1, 1
        if not max_q or nseq <= 0:
            return None
    assert block_tables.shape[0] >= nseq
    ws = torch.empty((_latr_ws(T, H, P, R, splits),), dtype=torch.uint8, device=q.device)
    out = torch.empty((T, H, E), dtype=q.dtype, device=q.device)
    _check(_latr(qp, q_row, dp, dkv_row, _f32(norm_w).data_ptr(), eps, _i32(positions).data_ptr(), _f32(inv_freq).data_ptr(),
                 int(rot_dims), int(neighbours), float(mult), cp, _i32(slot_mapping).data_ptr(), kp, vp,
                 block_tables.data_ptr(), block_tables.stride(0), k_cache.shape[1],
                 None if cu_q is None else _i32c(cu_q).data_ptr(), None if cu_q is not None else _i32c(lens).data_ptr(),
                 None if sink is None else _f32(sink).data_ptr(), ws.data_ptr(), out.data_ptr(), float(scale), T, nseq,
                 int(max_q), H, D, P, R, E, int(window), splits, _stream()), "latent_rows")
    return out


def latent_formed_rows(seqs: int, max_k: int) -> int:
    """Rows of formed keys and values that hold any ``seqs`` contexts of up to ``max_k`` tokens, each
    rounded up to whole tiles of 32."""
    return seqs * (-(-int(max_k) // 32) * 32)


def latent_formed_ok(q, dkv, up_k, up_v, k_cache, block_tables, seqs, max_q, max_k) -> bool:
    """Whether prompt portions run with their keys and values formed: bfloat16, sizes the kernels
    have (ranks of up to 512: ``latent_attention_ok``, whose weights are held in as many bits), pages of whole tiles of 32, and formed rows that take no more memory than the absorbed
    queries and the sums of latents of the other form do.  With that a context is at most 2 R / (D + E)
    times (R 512, D = E = 128: four times) the step's new tokens, sequence by sequence as long as the longest.
    On that line the forming pays too: us, absorbed / formed, 16 heads, R 512, 512 tokens behind 1536 146 / 100, 64 behind 192
    42.8 / 39.9, 8 times 32 behind 96 44.4 / 41.0; 16 tokens alone 29.5 / 29.5.  Beyond it a token forms more than it saves, and
    for R 128, where the two come out alike (8 prompts of about 1024: 109.6 / 108.7), the line lies at contexts without a prefix."""
    T, H, width = q.shape
    _, D, R = up_k.shape
    E, P = up_v.shape[2], width - D
    # (what turns most steps down first: a layer whose ranks are too low for it asks here on every prompt step)
    if not (max_q and max_k and seqs > 0 and T > 0) or max_q > max_k \
            or latent_formed_rows(seqs, max_k) * (D + E) > 2 * T * R:
        return False
    if any(t is None or t.dtype != torch.bfloat16 for t in (q, dkv, up_k, up_v, k_cache)) \
            or P <= 0 or dkv.shape[1] != R + P:
        return False
    return bool(k_cache.is_contiguous() and up_k.is_contiguous() and up_v.is_contiguous() and q.stride(2) == 1
                and q.stride(1) == width and width % 8 == 0 and (T == 1 or q.stride(0) % 8 == 0)
                and block_tables is not None and block_tables.dtype == torch.int32 and block_tables.stride(1) == 1
                and all(t.data_ptr() % 16 == 0 for t in (q, up_k, up_v, k_cache))
                and _latf_ok(D, E, R, P, k_cache.shape[1], block_tables.stride(0)))


def latent_formed_prompts(q, q_rot, k_cache, up_k, up_v, cu_q, block_tables, positions, scale, sink, max_q, max_k,
                          window=0, store=None):
    """``q`` [T, H, D + P] (the D-parts are read), ``q_rot`` [T, H, P] turned, cache rows [c | r] of the
    step's tokens already stored; sequence b owns rows cu_q[b] .. cu_q[b+1] and block table row b.
    Returns [T, H, E] (rows of no sequence hold anything).  ``store`` = (dkv, norm weight, eps, inv_freq, rot_dims,
    slot_mapping, neighbours, mult): the rows are stored and the queries turned here (``latent_rope_store``)."""
    T, H, width = q.shape
    D, R, E = up_k.shape[1], up_k.shape[2], up_v.shape[2]
    P, nseq = width - D, cu_q.shape[0] - 1
    rows = latent_formed_rows(nseq, max_k)
    nk, nv = -(-H * rows * D // 128) * 128, -(-H * rows * E // 128) * 128          # (on 256 bytes)
    ws = torch.empty((nk + nv + (T * H * P if store is not None else 0),), dtype=q.dtype, device=q.device)
    out = torch.empty((T, H, E), dtype=q.dtype, device=q.device)
    k, es, stream = ws.data_ptr(), ws.element_size(), _stream()
    if store is None:
        assert q_rot.shape == (T, H, P) and q_rot.is_contiguous()
        qr = q_rot.data_ptr()
    else:
        dkv, w, eps, inv_freq, rot_dims, slot_mapping, neighbours, mult = store
        assert dkv.dtype == q.dtype and q.stride(2) == 1 and q.stride(1) == width and dkv.stride(1) == 1 \
            and dkv.shape == (T, R + P) and w.numel() == R and inv_freq.numel() * 2 == rot_dims
        assert k_cache.is_contiguous() and k_cache.dtype == q.dtype and k_cache.shape[2:] == (1, R + P)
        qr = k + (nk + nv) * es
        _check(_lrs(None, q.data_ptr(), _rows(q), dkv.data_ptr(), _rows(dkv), _f32(w).data_ptr(), eps,
                    _i32(positions).data_ptr(), _f32(inv_freq).data_ptr(), int(rot_dims), k_cache.data_ptr(), None,
                    _ptr(_i32(slot_mapping)), qr, T, H, D, P, R, int(neighbours), float(mult), _dt(q), stream),
               "latent_rope_store")
    assert block_tables.shape[0] >= nseq
    _check(_latf(q.data_ptr(), q.stride(0), width, qr, H * P, k_cache.data_ptr(),
                 block_tables.data_ptr(), block_tables.stride(0), k_cache.shape[1], _i32c(cu_q).data_ptr(),
                 _i32(positions).data_ptr(), up_k.data_ptr(), up_v.data_ptr(), _ptr(_f32(sink)) if sink is not None else None,
                 k, k + nk * es, rows, out.data_ptr(), float(scale), nseq, int(max_q), H, D, E, R,
                 P, int(window), stream), "latent_formed_prompts")
    return out


def xielu(u, ap, aq, out_dtype):
    T, n = u.shape
    assert u.stride(1) == 1 and u.dtype == out_dtype
    act = torch.empty((T, n), dtype=out_dtype, device=u.device)
    _check(_xie(u.data_ptr(), _rows(u), act.data_ptr(), T, n, float(ap), float(aq), _dt(u),
                _stream()), "xielu")
    return act


def gated_group_norm(o, skip_x, skip_w, z, w, groups, eps, out_dtype):
    T, H, E = o.shape
    assert skip_x.shape == o.shape and z.shape == (T, H * E) and z.stride(1) == 1 \
        and z.dtype == out_dtype and w.numel() == H * E and skip_w.numel() == H
    out = torch.empty((T, H * E), dtype=out_dtype, device=o.device)
    _check(_ggn(_f32(o).data_ptr(), _f32(skip_x).data_ptr(), _f32(skip_w).data_ptr(), z.data_ptr(),
                _rows(z), _f32(w).data_ptr(), out.data_ptr(), T, H, E, int(groups), eps,
                _DT[out_dtype], _stream()), "gated_group_norm")
    return out


def sigmoid_gate(o, gate, out_dtype):
    T, H, E = o.shape
    assert o.stride(2) == 1 and gate.shape == (T, H * E) and gate.stride(1) == 1 \
        and o.dtype == out_dtype and gate.dtype == out_dtype
    out = torch.empty((T, H * E), dtype=out_dtype, device=o.device)
    _check(_sgt(o.data_ptr(), o.stride(0), o.stride(1), gate.data_ptr(), _rows(gate), out.data_ptr(),
                T, H, E, _dt(o), _stream()), "sigmoid_gate")
    return out


# ------------------------------------------------------------------ rotated values, pooled blocks
def half_rope_store(q, k, v, positions, inv_freq, rot_dims, v_inv_freq, k_cache, v_cache, slot_mapping):
    T, H, D = q.shape
    G, E = v.shape[1], v.shape[2]
    rs = q.stride(0)
    assert (T == 1 or (k.stride(0) == rs and v.stride(0) == rs)) and q.stride(1) == D \
        and k.stride(1) == D and v.stride(1) == E and q.stride(2) == 1, \
        "q / k / v must be views of one projection output"
    if k_cache is not None:
        assert k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.dtype == q.dtype \
            and k_cache.shape[2:] == (G, D) and v_cache.shape[2:] == (G, E)
    if rot_dims:
        assert inv_freq.numel() * 2 == rot_dims
    if v_inv_freq is not None:
        assert v_inv_freq.numel() * 2 == E
    _check(_hrs(q.data_ptr(), k.data_ptr(), v.data_ptr(), rs if T > 1 else int(rs or 0),
                _i32(positions).data_ptr(), _ptr(_f32(inv_freq)) if rot_dims else None, int(rot_dims),
                _ptr(_f32(v_inv_freq)) if v_inv_freq is not None else None, _ptr(k_cache), _ptr(v_cache),
                _ptr(_i32(slot_mapping)), T, H, G, D, E, _dt(q), _stream()), "half_rope_store")


def pool_block_means(k_cache, v_cache, k_pool, v_pool, pool, positions, block_tables, row_seq,
                     slot_mapping):
    n, bs, G, D = k_cache.shape
    E = v_cache.shape[3]
    T = positions.shape[0] if row_seq is None else min(positions.shape[0], row_seq.shape[0])
    assert k_cache.is_contiguous() and v_cache.is_contiguous() and k_pool.is_contiguous() \
        and v_pool.is_contiguous() and k_pool.dtype == k_cache.dtype and v_pool.dtype == k_cache.dtype
    assert block_tables.dtype == torch.int32 and block_tables.stride(1) == 1
    if row_seq is None:
        assert block_tables.shape[0] >= T
    _check(_pbm(k_cache.data_ptr(), v_cache.data_ptr(), k_pool.data_ptr(), v_pool.data_ptr(),
                _i32(positions).data_ptr(), _i32(slot_mapping).data_ptr(), block_tables.data_ptr(),
                block_tables.stride(0), _ptr(_i32(row_seq)), T, bs, int(pool), k_pool.shape[1], G, D, E,
                _dt(k_cache), _stream()), "pool_block_means")


def unturn_gate(o, positions, v_inv_freq, gate, out_dtype):
    T, H, E = o.shape
    assert o.stride(2) == 1 and o.dtype == out_dtype
    if gate is not None:
        assert gate.shape == (T, H * E) and gate.stride(1) == 1 and gate.dtype == out_dtype
    if v_inv_freq is not None:
        assert v_inv_freq.numel() * 2 == E
    out = torch.empty((T, H * E), dtype=out_dtype, device=o.device)
    _check(_utg(o.data_ptr(), o.stride(0), o.stride(1), _i32(positions).data_ptr(),
                _ptr(_f32(v_inv_freq)) if v_inv_freq is not None else None, _ptr(gate),
                _rows(gate) if gate is not None else 0, out.data_ptr(), T, H, E, _dt(o), _stream()),
           "unturn_gate")
    return out


# ------------------------------------------------------------------ real-gated diagonal recurrence
def short_conv(x, w, bias, conv_state, cu_q, positions, slots, row_seq):
    T, C = x.shape
    taps = _f32(w).shape[1]
    assert x.stride(1) == 1 and w.shape[0] == C
    if cu_q is not None:
        assert row_seq is not None, "prefill-form steps pass the sequence of each row"
    if taps > 1:
        assert _f32(conv_state).shape[1:] == (taps - 1, C)
    u = torch.empty((T, C), dtype=torch.float32, device=x.device)
    B = slots.shape[0]
    _check(_scv(x.data_ptr(), _rows(x), w.data_ptr(), _ptr(_f32(bias)) if bias is not None else None,
                _ptr(conv_state) if taps > 1 else None, _ptr(_i32(cu_q)), _i32(positions).data_ptr(),
                _i32(slots).data_ptr(), _ptr(_i32(row_seq)) if cu_q is not None else None,
                u.data_ptr(), T, B, C, taps, _dt(x), _stream()), "short_conv")
    return u


def scan_waves(rows: int, seqs: int, channels: int) -> int:
    """Parts a sequence's rows are cut into by the recurrence kernel (one wave each): enough
    workgroups x waves to fill the chip, parts of at least 32 rows."""
    per_seq = max(1, rows // max(seqs, 1))
    want = max(1, 4096 // max(seqs * ((channels + 63) // 64), 1))
    return max(1, min(16, want, per_seq // 32))


def rglru_scan(u, gates, gate_bias, lam, y, state, cu_q, positions, slots, sharp, out_dtype):
    T, C = u.shape
    nb = gates.shape[0]
    assert _f32(u) is u and _f32(gates).shape == (nb, T, 2 * (C // nb)) and _f32(gate_bias).shape == (nb, 2 * (C // nb))
    assert y.shape == (T, C) and y.stride(1) == 1 and y.dtype == out_dtype and _f32(state).shape[1] == C
    out = torch.empty((T, C), dtype=out_dtype, device=u.device)
    B = slots.shape[0]
    nw = scan_waves(T, B, C) if cu_q is not None else 1
    _check(_lru(u.data_ptr(), gates.data_ptr(), gate_bias.data_ptr(), _f32(lam).data_ptr(),
                y.data_ptr(), _rows(y), state.data_ptr(), _ptr(_i32(cu_q)), _i32(positions).data_ptr(),
                _i32(slots).data_ptr(), out.data_ptr(), T, B, C, nb, float(sharp), nw, _DT[out_dtype],
                _stream()), "rglru_scan")
    return out


def capped_glu_route_scale(gu, dense, ff, shared_ff, limit, shared_limit, out_dtype, slope=1.702,
                           shared_gate=True):
    T = gu.shape[0]
    C = gu.shape[1] // 2
    NR = dense.shape[1]
    NE = (C - shared_ff) // ff if ff else 0
    assert gu.stride(1) == 1 and gu.dtype == out_dtype and C == NE * ff + shared_ff and NR in (NE, NE + 1)
    act = torch.empty((T, C), dtype=out_dtype, device=gu.device)
    _check(_cgl(gu.data_ptr(), _rows(gu), _f32(dense).data_ptr(), act.data_ptr(), T, NE, NR, ff,
                shared_ff, float(limit), float(shared_limit), float(slope),
                int(bool(shared_gate) and NR > NE), _dt(gu), _stream()),
           "capped_glu_route_scale")
    return act


# ------------------------------------------------------------------ several residual streams
def _streams_of(x):
    """(streams, elements from one stream of a token to the next); rows dense."""
    assert x.dtype == torch.float32 and x.dim() == 3 and x.stride(2) == 1
    return x.shape[1], (x.stride(1) if x.shape[1] > 1 else x.shape[2])


def _norm_ptrs(read, norm, S, W):
    if read is None:
        return (None,) * 4
    alpha, w, b = norm
    assert read.numel() == S and w.numel() == W and b.numel() == W and alpha.numel() == 1
    return tuple(_f32(t).data_ptr() for t in (read, alpha, w, b))


def hyper_norm(x, read, norm, out_dtype):
    T, S, W = x.shape
    _, xs = _streams_of(x)
    h = torch.empty((T, W), dtype=out_dtype, device=x.device)
    _check(_hyp(x.data_ptr(), x.stride(0), xs, None, None, 0, None, 0, None, 0, None, None,
                *_norm_ptrs(read, norm, S, W), h.data_ptr(), T, S, W, _DT[out_dtype], _stream()),
           "hyper_norm")
    return h


def hyper_update_norm(x, y, skip, write, mix, read, norm, out_dtype):
    T, S, W = x.shape
    _, xs = _streams_of(x)
    assert y.shape == (T, W) and y.stride(1) == 1 and y.dtype == out_dtype
    assert write.numel() == S and mix.shape == (S, S)
    hs = gs = None
    if skip is not None:
        hs, gs = skip
        assert hs.shape == (T, W) and hs.stride(1) == 1 and hs.dtype == out_dtype
        assert gs.shape == (T,) and gs.dtype == torch.float32
    in_place = x.is_contiguous()
    new = x if in_place else torch.empty((T, S, W), dtype=torch.float32, device=x.device)
    h = torch.empty((T, W), dtype=out_dtype, device=x.device) if read is not None else None
    _check(_hyp(x.data_ptr(), x.stride(0) if not in_place else S * W, xs, new.data_ptr(), y.data_ptr(),
                _rows(y), _ptr(hs), _rows(hs) if hs is not None else 0, _ptr(gs),
                gs.stride(0) if gs is not None else 0, _f32(write).data_ptr(), _f32(mix).data_ptr(),
                *_norm_ptrs(read, norm, S, W), _ptr(h), T, S, W, _DT[out_dtype], _stream()),
           "hyper_update_norm")
    return new, h


def corrected_route(h, router_w, correction, top, identity, scale):
    T, W = h.shape
    NR = router_w.shape[0]
    assert h.is_contiguous() and router_w.shape[1] == W and correction.numel() == NR and 0 <= identity <= NR
    dense = torch.empty((T, NR - identity + 1), dtype=torch.float32, device=h.device)
    _check(_cor(h.data_ptr(), _f32(router_w).data_ptr(), _f32(correction).data_ptr(), dense.data_ptr(),
                T, W, NR - identity, NR, int(top), float(scale), _dt(h), _stream()), "corrected_route")
    return dense


def gelu_tanh_glu(gu, out_dtype):
    T, C = gu.shape[0], gu.shape[1] // 2
    assert gu.stride(1) == 1 and gu.dtype == out_dtype and gu.shape[1] == 2 * C
    act = torch.empty((T, C), dtype=out_dtype, device=gu.device)
    _check(_gtg(gu.data_ptr(), _rows(gu), act.data_ptr(), T, C, _dt(gu), _stream()), "gelu_tanh_glu")
    return act


# ------------------------------------------------------------------ filtered heads, token shift, wkv
def conv_norm_store(x, sizes, conv_w, conv_state, qw, kw, eps, k_cache, v_cache, slot_mapping, cu_q,
                    positions, slots, row_seq=None):
    H, G, D, E = sizes
    T, C = x.shape[0], (H + G) * D + G * E
    taps = _f32(conv_w).shape[1]
    assert x.stride(1) == 1 and x.shape[1] >= C and conv_w.shape[0] == C and qw.numel() == D and kw.numel() == D
    if cu_q is not None:
        assert row_seq is not None and row_seq.shape[0] >= T, "prefill-form steps pass the sequence of each row"
    if taps > 1:
        assert _f32(conv_state).shape[1:] == (taps - 1, C)
    if k_cache is not None:
        assert k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.dtype == x.dtype \
            and v_cache.dtype == x.dtype and k_cache.shape[2:] == (G, D) and v_cache.shape[2:] == (G, E)
    assert positions.shape[0] >= T and (slot_mapping is None or slot_mapping.shape[0] >= T)
    q = torch.empty((T, H, D), dtype=x.dtype, device=x.device)
    _check(_cns(x.data_ptr(), _rows(x), conv_w.data_ptr(), _ptr(conv_state) if taps > 1 else None,
                _f32(qw).data_ptr(), _f32(kw).data_ptr(), eps, q.data_ptr(), _ptr(k_cache), _ptr(v_cache),
                _ptr(_i32(slot_mapping)), _ptr(_i32(cu_q)), _i32(positions).data_ptr(),
                _i32(slots).data_ptr(), _ptr(_i32(row_seq)) if cu_q is not None else None, T,
                slots.shape[0], H, G, D, E, taps, _dt(x), _stream()), "conv_norm_store")
    return q


def shift_mix(h, mu, state, cu_q, positions, slots, row_seq=None):
    T, W = h.shape
    n = _f32(mu).shape[0]
    assert h.is_contiguous() and mu.shape[1] == W and _f32(state).shape[1:] == (1, W) and positions.shape[0] >= T
    if cu_q is not None:
        assert row_seq is not None and row_seq.shape[0] >= T, "prefill-form steps pass the sequence of each row"
    out = torch.empty((n, T, W), dtype=h.dtype, device=h.device)
    _check(_smx(h.data_ptr(), mu.data_ptr(), state.data_ptr(), _ptr(_i32(cu_q)), _i32(positions).data_ptr(),
                _i32(slots).data_ptr(), _ptr(_i32(row_seq)) if cu_q is not None else None, out.data_ptr(), T,
                slots.shape[0], W, n, _dt(h), _stream()), "shift_mix")
    return out


def wkv_scan(r, k, v, w_raw, w_bias, bonus, state, cu_q, positions, slots, longest=0):
    T, H, D = r.shape
    E, B = v.shape[2], slots.shape[0]
    assert state.shape[1:] == (H, D, E) and w_raw.shape == (T, H * D) and w_raw.stride(1) == 1
    assert k.dtype == r.dtype and v.dtype == r.dtype and w_raw.dtype == r.dtype
    assert w_bias.numel() == H * D and bonus.numel() == H * D
    if cu_q is not None and (T >= 96 * B or 2 * (longest or 0) >= 192 + B):
        o = _channel_chunks(1, r, k, v, w_raw, w_bias, _f32(bonus), 1.0, 1.0, state, cu_q, positions, slots,
                            int(longest or 0))
        if o is not None:
            return o
    o = _rows_out(T, H, E, slots, r.device)
    _check(_wkv(r.data_ptr(), k.data_ptr(), v.data_ptr(), _heads_view(r, D), _heads_view(k, D),
                _heads_view(v, E), w_raw.data_ptr(), _rows(w_raw), _f32(w_bias).data_ptr(),
                _f32(bonus).data_ptr(), _f32(state).data_ptr(), _ptr(_i32(cu_q)),
                _i32(positions).data_ptr(), _i32(slots).data_ptr(), o.data_ptr(), T, B, H, D, E,
                _dt(r), _stream()), "wkv_scan")
    return o


# ------------------------------------------------------------------ squared relu, token input of a layer
def relu_squared(u, out_dtype):
    T, n = u.shape
    assert u.stride(1) == 1 and u.dtype == out_dtype
    act = torch.empty((T, n), dtype=out_dtype, device=u.device)
    _check(_rsq(u.data_ptr(), _rows(u), act.data_ptr(), T, n, _dt(u), _stream()), "relu_squared")
    return act


def token_gate(z, ids, table, offset, out_dtype):
    T, n = z.shape
    assert z.stride(1) == 1 and z.dtype == out_dtype and table.dtype == out_dtype and table.stride(1) == 1
    assert ids.shape[0] >= T and 0 <= offset and offset + n <= table.shape[1]
    out = torch.empty((T, n), dtype=out_dtype, device=z.device)
    _check(_tgt(z.data_ptr(), _rows(z), _i32(ids).data_ptr(), table.data_ptr(), table.stride(0), int(offset),
                out.data_ptr(), T, n, _dt(z), _stream()), "token_gate")
    return out
