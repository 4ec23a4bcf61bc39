"""The memory a hybrid engine leaves free of KV blocks: what its mixers take beside a step's activations."""
import random

import pytest
import torch

import natilix_fixtures as fx
from test_natilix_engine import make_engine

from minivllm_amd.ops import hip_hybrid as hk


@pytest.mark.parametrize("tokens,seqs", [(16384, 256), (4096, 512), (1100, 512), (64, 8), (19, 4), (1, 1), (2000, 2000)])
def test_no_step_takes_more(tokens, seqs):
    shape = (32, 16, 128, 128)
    most = hk.delta_scan_workspace(tokens, seqs, *shape)
    r, top = random.Random(tokens), 0
    steps = [(tokens, b) for b in range(1, min(seqs, tokens) + 1)]
    steps += [(t, r.randint(1, min(seqs, t))) for t in (r.randint(1, tokens) for _ in range(2000))]
    for t, b in steps:
        top = max(top, hk._scan_ws(256, 256, 256, 256, 256, t, b, *shape))
    assert most == top


def test_blocks_leave_room(tmp_path, monkeypatch):
    """A card of 1 GiB whose free memory a chunked delta rule's workspace takes a good part of."""
    c = fx.config([(fx.delta(heads=4, kv_heads=2, dim=16, vdim=16), None), (fx.attention(), None)])
    eng = make_engine(tmp_path, c, fx.weights(c), "cpu", "float32")
    run = eng.model_runner
    run.cfg.max_cached_blocks, run.cfg.max_num_batched_tokens, run.cfg.max_num_sequences = None, 32768, 512
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda: (1 << 30, 1 << 30))
    monkeypatch.setattr(torch.cuda, "memory_stats", lambda: {})
    monkeypatch.setattr(type(run), "_allocate_hybrid_caches", lambda self: None)
    run.on_gpu = True
    run.allocate_kv_cache()
    workspace = hk._scan_ws(256, 256, 256, 256, 256, 32768, 512, 4, 2, 16, 16)
    assert workspace > 100 << 20
    left = int((1 << 30) * run.cfg.gpu_memory_utilization) - run.num_kv_blocks * run.kv_block_bytes()
    assert left >= workspace + run._state_bytes() + 32768 * run._widest_row_bytes()
