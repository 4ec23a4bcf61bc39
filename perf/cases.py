"""Workloads of this engine, each a call (or a short run of calls) through its public entry points:
the attention functions of the dense decoders (``layers.attention``, ``ops``), the mixers of the
hybrid decoders as a model calls them (``layers``), and whole requests through ``LLMEngine``.

``listed()`` names the workloads, ``draw(rng)`` gives further ones of the same ranges, ``prepare``
makes what a program holds before the call, ``run`` is one pass, ``exact`` the same outputs in 64
bits with plain torch, ``work`` the bytes and operations of a pass and ``tolerance`` how far two
correct implementations of one precision may lie apart.

Head geometries, widths, lengths and batch sizes are those of the repository's benchmarks
(``benchmark_decoding.py``, ``benchmark_prefilling.py``, ``benchmark_models.py``, ``bench.py`` and its
``--hybrid`` sizes) and test configurations.
"""
import math
import random

import torch

DEV = "cuda"
F64 = torch.float64
DT = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
EPS = 1e-6


# ------------------------------------------------------------------ the cases
def _decode(name, **kw):
    return dict({"name": name, "kind": "decode", "dtype": "bf16", "batch": 1, "context": 512, "ragged": True,
                 "heads": 32, "kv_heads": 8, "dim": 128, "block": 256, "fp8": False}, **kw)


def _prefill(name, **kw):
    return dict({"name": name, "kind": "prefill", "dtype": "bf16", "seqs": 1, "length": 512, "ragged": True,
                 "heads": 32, "kv_heads": 8, "dim": 128, "block": 256, "paged": True, "prefix": 0}, **kw)


def _request(name, **kw):
    return dict({"name": name, "kind": "request", "prompts": 4, "length": 256, "steps": 8}, **kw)


def _attention(name, **kw):
    return dict({"name": name, "kind": "attention", "phase": "prefill", "dtype": "bf16", "seqs": 8, "length": 1024,
                 "ragged": True, "heads": 16, "kv_heads": 8, "dim": 128, "vdim": 128, "window": 0,
                 "keep_first": 0, "chunk": 0, "sink": True, "gate": True, "slopes": False, "prefix": 0,
                 "block": 256}, **kw)


def _latent(name, **kw):
    return dict({"name": name, "kind": "latent", "phase": "prefill", "dtype": "bf16", "seqs": 8, "length": 1024,
                 "ragged": True, "heads": 16, "dim": 128, "rot": 64, "rank": 512, "vdim": 128, "window": 0,
                 "sink": False, "block": 256}, **kw)


def _delta(name, **kw):
    return dict({"name": name, "kind": "delta", "phase": "prefill", "dtype": "bf16", "seqs": 8, "length": 1024,
                 "ragged": True, "heads": 16, "kv_heads": 8, "dim": 128, "vdim": 128, "conv": 4,
                 "channel": False, "past": False}, **kw)


def _scan(name, **kw):
    return dict({"name": name, "kind": "scan", "rule": "gla", "phase": "prefill", "dtype": "bf16", "seqs": 8,
                 "length": 1024, "ragged": True, "heads": 8, "dim": 64, "vdim": 128, "past": False}, **kw)


def listed():
    return [
        # one user's next token over a short context in the reference's cache layout (fp16, blocks of 16
        # tokens): nothing but latency
        _decode("decode_one", dtype="fp16", batch=1, context=512, ragged=False, block=16),
        # a serving batch's next tokens: the KV cache is streamed once
        _decode("decode_batch", batch=256, context=1024),
        # two short chat prompts, packed keys and values
        _prefill("prefill_short", dtype="fp16", seqs=2, length=60, ragged=False, paged=False),
        # a serving prefill step: 16 prompts of mixed length through the block table
        _prefill("prefill_batch", seqs=16, length=1024),
        # whole requests of the dense decoder through the engine: prompts, then tokens one by one
        _request("request_dense", prompts=4, length=256, steps=8),
        # hybrid decoder, softmax attention layer with sink and gate: 8 prompts of about 1k tokens
        _attention("attention_prompts"),
        # the same layer kind with a window and kept first tokens in a 32-bit engine, odd lengths
        _attention("attention_window_fp32", dtype="fp32", seqs=3, length=611, window=256, keep_first=4, gate=False,
                   sink=False, heads=8, kv_heads=4, dim=64, vdim=64),
        # its next tokens for 64 running sequences
        _attention("attention_next", phase="decode", seqs=64, length=1024),
        # latent attention layer (low-rank keys and values), 8 prompts of about 1k tokens
        _latent("latent_prompts"),
        # gated delta rule layer, 8 prompts of about 1k tokens
        _delta("delta_prompts"),
        # its next tokens for 64 running sequences: the state is read and written once
        _delta("delta_next", phase="decode", seqs=64),
        # matrix LSTM layer, 8 prompts of about 1k tokens
        _scan("mlstm_prompts", rule="mlstm", dim=128),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["decode", "prefill", "request", "attention", "attention", "latent", "delta", "scan"])
    if kind == "decode":
        batch = _log(rng, 1, 256)
        h, g, d = rng.choice([(32, 8, 128), (16, 8, 128), (40, 8, 128), (64, 8, 128), (28, 4, 128), (4, 2, 64)])
        c = _decode("", dtype=rng.choice(["bf16", "fp16"]), batch=batch,
                    context=_log(rng, 16, min(8192, 262144 // batch)), heads=h, kv_heads=g, dim=d,
                    block=rng.choice([16, 64, 256]), fp8=rng.random() < 0.25, ragged=rng.random() < 0.8)
    elif kind == "prefill":
        seqs = _log(rng, 1, 16)
        h, g, d = rng.choice([(32, 8, 128), (16, 8, 128), (40, 8, 128), (28, 4, 128), (4, 2, 64)])
        paged = rng.random() < 0.6
        c = _prefill("", dtype=rng.choice(["bf16", "fp16"]), seqs=seqs, length=_log(rng, 16, min(4096, 16384 // seqs)),
                     heads=h, kv_heads=g, dim=d, block=rng.choice([16, 64, 256]), paged=paged,
                     prefix=_log(rng, 16, 512) if paged and rng.random() < 0.4 else 0, ragged=rng.random() < 0.8)
    elif kind == "request":
        prompts = rng.randint(1, 8)
        c = _request("", prompts=prompts, length=_log(rng, 16, min(600, 1024 // prompts)), steps=rng.randint(1, 8))
    elif kind == "attention":
        phase = rng.choice(["prefill", "prefill", "decode"])
        seqs = _log(rng, 1, 128 if phase == "decode" else 8)
        h, g, d, e = rng.choice([(16, 8, 128, 128), (16, 8, 128, 128), (8, 4, 64, 64), (8, 2, 128, 64), (6, 3, 48, 40)])
        window = rng.choice([0, 0, 128, 512])
        chunk = rng.choice([0, 256]) if not window else 0
        c = _attention("", phase=phase, dtype=rng.choice(["bf16", "bf16", "fp32"]), seqs=seqs,
                       length=_log(rng, 16, min(2048, (131072 if phase == "decode" else 8192) // seqs)),
                       heads=h, kv_heads=g, dim=d, vdim=e, window=window, chunk=chunk,
                       keep_first=4 if window and rng.random() < 0.5 else 0, sink=rng.random() < 0.5,
                       gate=rng.random() < 0.5, slopes=not chunk and rng.random() < 0.25,
                       prefix=_log(rng, 16, 512) if phase == "prefill" and rng.random() < 0.3 else 0,
                       block=rng.choice([16, 64, 256]))
    elif kind == "latent":
        phase = rng.choice(["prefill", "decode"])
        seqs = _log(rng, 1, 128 if phase == "decode" else 8)
        rank, rot = rng.choice([(512, 64), (512, 64), (128, 128), (256, 64)])
        c = _latent("", phase=phase, seqs=seqs, length=_log(rng, 16, min(2048, (65536 if phase == "decode" else 8192) // seqs)),
                    heads=rng.choice([16, 16, 6]), rot=rot, rank=rank, window=rng.choice([0, 0, 512]),
                    sink=rng.random() < 0.5, block=rng.choice([64, 256]))
    elif kind == "delta":
        phase = rng.choice(["prefill", "prefill", "decode"])
        seqs = _log(rng, 1, 64 if phase == "decode" else 8)
        h, g, d, e = rng.choice([(16, 8, 128, 128), (16, 8, 128, 128), (8, 4, 64, 64), (4, 2, 48, 40)])
        c = _delta("", phase=phase, dtype=rng.choice(["bf16", "bf16", "fp32"]), seqs=seqs,
                   length=_log(rng, 4, 1024), heads=h, kv_heads=g, dim=d, vdim=e,
                   conv=rng.choice([4, 4, 2]), channel=rng.random() < 0.4, past=rng.random() < 0.3)
    else:
        phase = rng.choice(["prefill", "prefill", "decode"])
        seqs = _log(rng, 1, 64 if phase == "decode" else 8)
        rule = rng.choice(["gla", "mlstm", "wkv"])
        h, d, e = {"gla": (8, 64, 128), "mlstm": (8, 128, 128), "wkv": (16, 64, 64)}[rule]
        if rng.random() < 0.3:
            h, d, e = (4, 48, 48) if rule == "wkv" else (4, 48, 40)
        c = _scan("", rule=rule, phase=phase, dtype=rng.choice(["bf16", "bf16", "fp32"]), seqs=seqs,
                  length=_log(rng, 4, 1024), heads=h, dim=d, vdim=e, past=rng.random() < 0.3)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs
def _lengths(c, n, longest):
    """The sequences' lengths: a property of the case, not of the seed."""
    if not c.get("ragged"):
        return [longest] * n
    r = random.Random("%s %d %d %s" % (c["kind"], n, longest, c.get("phase", "")))
    out = [max(1, round(longest * r.uniform(0.5, 1.0))) for _ in range(n)]
    out[r.randrange(n)] = longest
    return out


def _layout(c):
    """(new tokens per sequence, tokens already there per sequence)."""
    if c["kind"] == "decode":
        return [1] * c["batch"], [n - 1 for n in _lengths(c, c["batch"], c["context"])]
    lens = _lengths(c, c["seqs"], c["length"])
    if c.get("phase") == "decode":
        return [1] * len(lens), [n - 1 for n in lens]
    if c["kind"] in ("delta", "scan"):
        return lens, [37 if c["past"] else 0] * len(lens)
    return lens, [c["prefix"] if "prefix" in c else 0] * len(lens)


class _Maker:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)
        self.r = random.Random(seed)

    def randn(self, *shape, dtype=torch.float32, std=1.0, mean=0.0):
        return (torch.randn(*shape, generator=self.g, device=DEV) * std + mean).to(dtype)

    def uniform(self, lo, hi, *shape):
        return torch.rand(*shape, generator=self.g, device=DEV) * (hi - lo) + lo


def _ints(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def _cum(lens):
    out = [0]
    for n in lens:
        out.append(out[-1] + n)
    return out


def _pages(m, totals, block):
    """Block tables over pages in no particular order; the number of pages."""
    need = [-(-n // block) for n in totals]
    ids = list(range(sum(need)))
    m.r.shuffle(ids)
    width, rows, at = max(need), [], 0
    for n in need:
        rows.append(ids[at:at + n] + [0] * (width - n))
        at += n
    return _ints(rows), len(ids)


def _slot_mapping(tables, new, past, block):
    """The cache slot of every new token."""
    t = tables.tolist()
    return _ints([t[b][p // block] * block + p % block
                  for b, (n, s) in enumerate(zip(new, past)) for p in range(s, s + n)])


def _context_of(c, new, past, tables, block=0):
    """What the engine tells the layers about a step."""
    B = len(new)
    pos = [s + i for n, s in zip(new, past) for i in range(n)]
    kw = dict(positions=_ints(pos), num_seqs=B, block_tables=tables, state_slots=_ints(list(range(B))[::-1]))
    if tables is not None:
        kw["slot_mapping"] = _slot_mapping(tables, new, past, block)
    total = [n + s for n, s in zip(new, past)]
    if c["phase"] == "decode":
        kw.update(context_lens=_ints(total), max_context_len=max(total))
        return False, kw
    kw.update(cu_seqlens_q=_ints(_cum(new)), cu_seqlens_k=_ints(_cum(total)), max_seqlen_q=max(new),
              max_seqlen_k=max(total), row_seq=_ints([b for b, n in enumerate(new) for _ in range(n)]))
    return True, kw


def _fill(module, m, c):
    """Weights of a mixer with the spread that trained ones have."""
    w = {}
    for name, p in module.named_parameters():
        if name == "conv_weight":
            v = m.randn(*p.shape, std=0.4)
        elif name == "A_log":
            v = m.uniform(1.0, 16.0, *p.shape).log()
        elif name == "dt_bias":
            dt = m.uniform(math.log(1e-3), math.log(1e-1), *p.shape).exp()
            v = dt + torch.log(-torch.expm1(-dt))
        elif name == "f_bias":
            v = m.uniform(3.0, 6.0, *p.shape)
        elif name in ("norm_weight", "latent_norm"):
            v = m.randn(*p.shape, std=0.1, mean=1.0)
        elif name.startswith("up_"):
            v = m.randn(*p.shape, std=p.shape[1] ** -0.5)
        else:
            v = m.randn(*p.shape)
        p.data = v.to(p.dtype)
        w[name] = p.data
    return w


_ENGINE = []
DENSE = dict(vocab_size=32768, hidden_size=1024, num_heads=16, num_kv_heads=8, head_dim=128, intermediate_size=3072,
             num_layers=8, max_position=8192, tie_word_embeddings=False, name="dense-w1024")


def _dense_weight(name, shape, dtype=torch.bfloat16):
    """The engine's weights are the same whatever the requests are."""
    g = torch.Generator(device=DEV)
    g.manual_seed(sum(ord(ch) * (i + 1) for i, ch in enumerate(name)) % 1000003)
    if name.endswith("norm.weight"):
        if "layernorm" in name:
            return torch.ones(shape, dtype=dtype, device=DEV)
        return (1.0 + 0.1 * torch.randn(shape, generator=g, device=DEV)).to(dtype)
    return (torch.randn(shape, generator=g, device=DEV) * 0.03).to(dtype)


def _engine():
    """One engine serves all requests of a program.  (The start-up timing of GEMM variants is off, so
    that every start runs the same kernels.)"""
    if not _ENGINE:
        from minivllm_amd.config import ModelConfig
        from minivllm_amd.engine.llm_engine import LLMEngine
        eng = LLMEngine(dict(model=ModelConfig(**DENSE), max_num_sequences=8, max_num_batched_tokens=8192,
                             block_size=256, max_model_length=2048, max_cached_blocks=96, eos=-1, dtype="bfloat16",
                             device="cuda", graph_batch_sizes=[1, 2, 4, 8], prefill_graph_max_tokens=0,
                             tune_decode_gemms=False, tune_prefill_gemms=False, score_only=True))
        with torch.no_grad():
            for name, p in eng.model_runner.model.named_parameters():
                p.copy_(_dense_weight(name, p.shape, p.dtype))
        _ENGINE.append(eng)
    return _ENGINE[0]


def prepare(c, seed):
    m = _Maker(seed)
    return _PREPARE[c["kind"]](c, m, seed)


def _cache(m, pages, block, heads, dim, dtype, fp8=False):
    """[pages, block, heads, dim] in the engine's order: a page's tokens of one head lie together."""
    x = torch.randn(pages, heads, block, dim, generator=m.g, device=DEV, dtype=dtype)
    return (x.to(torch.float8_e4m3fn) if fp8 else x).permute(0, 2, 1, 3)


def _prepare_decode(c, m, seed):
    dt, (new, past) = DT[c["dtype"]], _layout(c)
    total = [n + s for n, s in zip(new, past)]
    tables, pages = _pages(m, total, c["block"])
    a = (pages, c["block"], c["kv_heads"], c["dim"], dt, c["fp8"])
    return dict(c=c, q=m.randn(c["batch"], c["heads"], c["dim"], dtype=dt), k=_cache(m, *a), v=_cache(m, *a),
                tables=tables, lens=_ints(total), longest=max(total), scale=c["dim"] ** -0.5)


def _prepare_prefill(c, m, seed):
    dt, (new, past) = DT[c["dtype"]], _layout(c)
    total = [n + s for n, s in zip(new, past)]
    T, G, D = sum(new), c["kv_heads"], c["dim"]
    st = dict(c=c, q=m.randn(T, c["heads"], D, dtype=dt), cu=_ints(_cum(new)), longest=max(new), scale=D ** -0.5)
    if c["paged"]:
        st["tables"], pages = _pages(m, total, c["block"])
        st.update(k=_cache(m, pages, c["block"], G, D, dt), v=_cache(m, pages, c["block"], G, D, dt),
                  cu_k=_ints(_cum(total)))
    else:
        st.update(k=m.randn(T, G, D, dtype=dt), v=m.randn(T, G, D, dtype=dt))
    return st


def _prepare_request(c, m, seed):
    lens = _lengths(dict(c, ragged=True), c["prompts"], c["length"])
    return dict(c=c, engine=_engine(), names=["%d-%d" % (seed, i) for i in range(len(lens))],
                prompts=[[m.r.randrange(DENSE["vocab_size"]) for _ in range(n)] for n in lens],
                given=[[m.r.randrange(DENSE["vocab_size"]) for _ in range(c["steps"])] for _ in lens])


def _prepare_attention(c, m, seed):
    from minivllm_amd.layers.attention import SinkAttention
    dt, (new, past) = DT[c["dtype"]], _layout(c)
    H, G, D, E = c["heads"], c["kv_heads"], c["dim"], c["vdim"]
    total = [n + s for n, s in zip(new, past)]
    tables, pages = _pages(m, total, c["block"])
    slopes = torch.tensor([2.0 ** (-8.0 * (h + 1) / H) for h in range(H)]) if c["slopes"] else None
    mod = SinkAttention(H, G, D, E, D ** -0.5, sink=c["sink"], window=c["window"], keep_first=c["keep_first"],
                        distance_slopes=slopes, chunk=c["chunk"]).to(DEV)
    w = _fill(mod, m, c)
    mod.k_cache = m.randn(pages, c["block"], G, D, dtype=dt)
    mod.v_cache = m.randn(pages, c["block"], G, E, dtype=dt)
    T = sum(new)
    # q and the gates are column blocks of one projection's output
    proj = m.randn(T, H * D + H, dtype=dt)
    return dict(c=c, mod=mod, w=w, ctx=_context_of(c, new, past, tables, c["block"]), q=proj[:, :H * D].view(T, H, D),
                gate=proj[:, H * D:] if c["gate"] else None)


def _prepare_latent(c, m, seed):
    from minivllm_amd.layers.attention import LatentAttention
    from minivllm_amd.layers.rotary_embedding import HalfRotation
    dt, (new, past) = DT[c["dtype"]], _layout(c)
    H, D, P, R, E = c["heads"], c["dim"], c["rot"], c["rank"], c["vdim"]
    total = [n + s for n, s in zip(new, past)]
    tables, pages = _pages(m, total, c["block"])
    mod = LatentAttention(H, D, P, E, R, (D + P) ** -0.5, c["window"], HalfRotation(P, 10000.0), EPS,
                          sink=c["sink"]).to(DEV)
    for name in ("up_k", "up_v"):
        setattr(mod, name, torch.nn.Parameter(getattr(mod, name).data.to(dt), requires_grad=False))
    w = _fill(mod, m, c)
    rows = m.randn(pages, c["block"], 1, R + P, dtype=dt)
    mod.core.k_cache = rows
    mod.core.v_cache = rows[..., :R]
    T = sum(new)
    return dict(c=c, mod=mod, w=w, ctx=_context_of(c, new, past, tables, c["block"]), q=m.randn(T, H, D + P, dtype=dt),
                dkv=m.randn(T, R + P, dtype=dt), rows=rows)


def _states(m, holder, B):
    for name, shape in holder.state_spec():
        setattr(holder, name, m.randn(B, *shape, std=0.2))


def _prepare_delta(c, m, seed):
    from minivllm_amd.layers.delta_rule import GatedDeltaRule
    dt, (new, past) = DT[c["dtype"]], _layout(c)
    H, D, E = c["heads"], c["dim"], c["vdim"]
    mod = GatedDeltaRule(H, c["kv_heads"], D, E, c["conv"], EPS, channel_decay=c["channel"]).to(DEV)
    w = _fill(mod, m, c)
    _states(m, mod, len(new))
    T = sum(new)
    st = dict(c=c, mod=mod, w=w, dt=dt, ctx=_context_of(c, new, past, None),
              proj=m.randn(T, sum(mod.split_sizes()), dtype=dt), a=None, gate=None)
    if c["channel"]:
        st.update(a=m.randn(T, H * D, dtype=dt), gate=m.randn(T, H * E, dtype=dt))
    return st


def _prepare_scan(c, m, seed):
    from minivllm_amd.layers.linear_attention import GatedLinearAttention, MatrixLSTM
    dt, (new, past) = DT[c["dtype"]], _layout(c)
    H, D, E = c["heads"], c["dim"], c["vdim"]
    T, B = sum(new), len(new)
    st = dict(c=c, dt=dt, ctx=_context_of(c, new, past, None))
    if c["rule"] == "wkv":
        st["w"] = dict(w_bias=m.uniform(-6.0, -1.0, H * D), bonus=m.randn(H, D, std=0.5),
                       norm_weight=m.randn(H * E, std=0.1, mean=1.0))
        st["state"] = m.randn(B, H, D, E, std=0.2)
        for x, n in (("r", D), ("k", D), ("v", E)):
            st[x] = m.randn(T, H, n, dtype=dt)
        st.update(w_raw=m.randn(T, H * D, dtype=dt, std=0.5), gate=m.randn(T, H * E, dtype=dt))
        return st
    if c["rule"] == "mlstm":
        mod = MatrixLSTM(H, D, E, 15.0, EPS).to(DEV)
    else:
        mod = GatedLinearAttention(H, D, E, 16.0, EPS).to(DEV)
        st["decay_raw"] = m.randn(T, H * D, dtype=dt)
    st.update(mod=mod, w=_fill(mod, m, c), proj=m.randn(T, sum(mod.split_sizes()), dtype=dt))
    _states(m, mod, B)
    if c["rule"] == "mlstm":          # every copy of a sequence's normaliser and maximum is the same
        mod.norm_state.copy_(mod.norm_state[:, :, :1].clone())
        mod.max_state.copy_(mod.max_state[:, :, :1].clone())
    return st


_PREPARE = dict(decode=_prepare_decode, prefill=_prepare_prefill, request=_prepare_request,
                attention=_prepare_attention, latent=_prepare_latent, delta=_prepare_delta, scan=_prepare_scan)


# ------------------------------------------------------------------ one pass
def run(st):
    return _RUN[st["c"]["kind"]](st, st["c"])


def _run_decode(st, c):
    from minivllm_amd.layers.attention import paged_attention_decode
    return paged_attention_decode(st["q"], st["k"], st["v"], st["tables"], st["lens"], st["scale"], c["heads"],
                                  c["kv_heads"], c["dim"], c["block"], st["longest"])


def _run_prefill(st, c):
    if c["paged"]:
        from minivllm_amd import ops
        return ops.paged_attention_prefill(st["q"], st["k"], st["v"], st["cu"], st["cu_k"], st["tables"], st["scale"],
                                           st["longest"])
    from minivllm_amd.layers.attention import flash_attention_prefill
    return flash_attention_prefill(st["q"], st["k"], st["v"], st["cu"], st["scale"], c["heads"], c["kv_heads"],
                                   c["dim"], st["longest"])


def _run_request(st, c):
    eng, names = st["engine"], st["names"]
    got = eng.score_step([{"id": n, "tokens": p, "want": [len(p) - 1]} for n, p in zip(names, st["prompts"])])
    out = [torch.cat([got[n] for n in names])]
    for s in range(c["steps"]):
        got = eng.score_step([{"id": n, "tokens": [g[s]], "want": [0]} for n, g in zip(names, st["given"])],
                             end=names if s == c["steps"] - 1 else ())
        out.append(torch.cat([got[n] for n in names]))
    return torch.stack(out)


def _in_step(st):
    from minivllm_amd.utils.context import set_context
    set_context(st["ctx"][0], **st["ctx"][1])


def _run_attention(st, c):
    _in_step(st)
    with torch.inference_mode():
        return st["mod"](st["q"], st["gate"])


def _run_latent(st, c):
    _in_step(st)
    with torch.inference_mode():
        return st["mod"](st["q"], st["dkv"])


def _run_delta(st, c):
    _in_step(st)
    with torch.inference_mode():
        y = st["mod"](st["proj"], st["dt"], st["a"], st["gate"])
    return dict(y=y, state=st["mod"].state, conv=st["mod"].conv_state)


def _run_scan(st, c):
    _in_step(st)
    with torch.inference_mode():
        if c["rule"] == "wkv":
            from minivllm_amd import ops
            pre, kw = st["ctx"]
            w = st["w"]
            o = ops.wkv_scan(st["r"], st["k"], st["v"], st["w_raw"], w["w_bias"], w["bonus"], st["state"],
                             kw["cu_seqlens_q"] if pre else None, kw["positions"], kw["state_slots"])
            y = ops.gated_head_norm(o, w["norm_weight"], st["gate"], EPS, st["dt"], "silu")
            return dict(y=y.view(y.shape[0], -1), state=st["state"])
        mod = st["mod"]
        if c["rule"] == "gla":
            return dict(y=mod(st["proj"], st["decay_raw"], st["dt"]), state=mod.state)
        return dict(y=mod(st["proj"], st["dt"]), state=mod.state, norm=mod.norm_state, top=mod.max_state)


_RUN = dict(decode=_run_decode, prefill=_run_prefill, request=_run_request, attention=_run_attention,
            latent=_run_latent, delta=_run_delta, scan=_run_scan)


# ------------------------------------------------------------------ the same in 64 bits
def exact(c, seed):
    m = _Maker(seed)
    if c["kind"] == "request":
        return _exact_request(c, m)
    return _EXACT[c["kind"]](c, _PREPARE[c["kind"]](c, m, seed))


def _gather(cache, row, n):
    """The first n tokens of a sequence: [n, heads, dim] in 64 bits."""
    bs = cache.shape[1]
    return cache[row[:-(-n // bs)].long()].reshape(-1, *cache.shape[2:])[:n].to(F64)


def _attend(q, k, v, scale, past, window=0, keep_first=0, chunk=0, sink=None, slopes=None):
    """q [n, H, D] at positions past .. past + n - 1 over k [m, G, D], v [m, G, E] -> [n, H, E]."""
    n, H, _ = q.shape
    r = H // k.shape[1]
    kt = k.transpose(0, 1).repeat_interleave(r, 0)
    vt = v.transpose(0, 1).repeat_interleave(r, 0)
    out = torch.empty(n, H, v.shape[2], dtype=F64, device=q.device)
    at = torch.arange(k.shape[0], device=q.device)[None]
    step = max(1, (1 << 27) // (H * k.shape[0]))
    for s in range(0, n, step):
        e = min(n, s + step)
        i = torch.arange(past + s, past + e, device=q.device)[:, None]
        z = torch.matmul(q[s:e].transpose(0, 1), kt.transpose(1, 2)) * scale
        if slopes is not None:
            z = z - slopes.to(F64)[:, None, None] * (i - at).to(F64)
        off = at > i
        if window:
            off = off | ((i - at >= window) & (at >= keep_first))
        if chunk:
            off = off | (i // chunk != at // chunk)
        z = z.masked_fill(off[None], -math.inf)
        if sink is not None:
            z = torch.cat([z, sink.to(F64)[:, None, None].expand(H, e - s, 1)], -1)
        out[s:e] = torch.matmul(torch.softmax(z, -1)[..., :k.shape[0]], vt).transpose(0, 1)
    return out


def _exact_decode(c, st):
    out = torch.empty(st["q"].shape, dtype=F64, device=DEV)
    for b, n in enumerate(st["lens"].tolist()):
        row = st["tables"][b]
        out[b:b + 1] = _attend(st["q"][b:b + 1].to(F64), _gather(st["k"], row, n), _gather(st["v"], row, n),
                               st["scale"], n - 1)
    return out


def _exact_prefill(c, st):
    new, past = _layout(c)
    out, at = torch.empty(st["q"].shape, dtype=F64, device=DEV), 0
    for b, (n, s) in enumerate(zip(new, past)):
        if c["paged"]:
            k, v = (_gather(st[x], st["tables"][b], n + s) for x in "kv")
        else:
            k, v = st["k"][at:at + n].to(F64), st["v"][at:at + n].to(F64)
        out[at:at + n] = _attend(st["q"][at:at + n].to(F64), k, v, st["scale"], s)
        at += n
    return out


def _exact_attention(c, st):
    new, past = _layout(c)
    mod, tables = st["mod"], st["ctx"][1]["block_tables"]
    out, at = [], 0
    for b, (n, s) in enumerate(zip(new, past)):
        o = _attend(st["q"][at:at + n].to(F64), _gather(mod.k_cache, tables[b], n + s),
                    _gather(mod.v_cache, tables[b], n + s), c["dim"] ** -0.5, s, c["window"], c["keep_first"],
                    c["chunk"], st["w"].get("sink"), mod.slopes)
        if st["gate"] is not None:
            o = o * torch.sigmoid(st["gate"][at:at + n].to(F64))[:, :, None]
        out.append(o.reshape(n, -1))
        at += n
    return torch.cat(out)


def _rms(x):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS)


def _half_turn(x, pos, dims, base):
    """Entries i and i + dims / 2 of the first ``dims`` turn together; x [T, heads, n]."""
    f = base ** (-torch.arange(0, dims, 2, dtype=F64, device=x.device) / dims)
    a = (pos.to(F64)[:, None] * f)[:, None]
    x1, x2 = x[..., :dims // 2], x[..., dims // 2:dims]
    return torch.cat([x1 * a.cos() - x2 * a.sin(), x2 * a.cos() + x1 * a.sin(), x[..., dims:]], -1)


def _exact_latent(c, st):
    new, past = _layout(c)
    D, P, R, w, kw = c["dim"], c["rot"], c["rank"], st["w"], st["ctx"][1]
    pos, rows = kw["positions"], st["rows"].to(F64)
    q, dkv = st["q"].to(F64), st["dkv"].to(F64)
    lat = torch.cat([_rms(dkv[:, :R]) * w["latent_norm"].to(F64),
                     _half_turn(dkv[:, None, R:], pos, P, 10000.0)[:, 0]], -1)
    rows.view(-1, R + P)[kw["slot_mapping"].long()] = lat
    qa = torch.cat([torch.einsum("thd,hdr->thr", q[..., :D], w["up_k"].to(F64)),
                    _half_turn(q[..., D:], pos, P, 10000.0)], -1)
    out, at = [], 0
    for b, (n, s) in enumerate(zip(new, past)):
        k = _gather(rows, kw["block_tables"][b], n + s)
        o = _attend(qa[at:at + n], k, k[..., :R], (D + P) ** -0.5, s, c["window"], sink=w.get("core.sink"))
        out.append(torch.einsum("thr,hre->the", o, w["up_v"].to(F64)))
        at += n
    return torch.cat(out)


def _padded(c, *xs):
    """Rows of a step -> [sequences, longest, ...] in 64 bits."""
    new, _ = _layout(c)
    got = []
    for x in xs:
        y = torch.zeros(len(new), max(new), *x.shape[1:], dtype=F64, device=DEV)
        at = 0
        for b, n in enumerate(new):
            y[b, :n] = x[at:at + n].to(F64)
            at += n
        got.append(y)
    return got


def _rows_of(c, y):
    return torch.cat([y[b, :n] for b, n in enumerate(_layout(c)[0])])


def _live(c, t):
    """Which sequences have a token t."""
    return torch.tensor([n > t for n in _layout(c)[0]], device=DEV)


def _first_state(c, st, x):
    """The state the sequences start from, in the order of the sequences."""
    slots = st["ctx"][1]["state_slots"].long()
    keep = torch.tensor([s > 0 for s in _layout(c)[1]], device=DEV)
    y = x[slots].to(F64)
    return torch.where(keep.view(-1, *[1] * (y.dim() - 1)), y, torch.zeros_like(y))


def _to_slots(st, x, like):
    out = like.to(F64).clone()
    out[st["ctx"][1]["state_slots"].long()] = x
    return out


def _exact_delta(c, st):
    new, past = _layout(c)
    mod, w, B = st["mod"], st["w"], len(new)
    H, G, D, E, taps = c["heads"], c["kv_heads"], c["dim"], c["vdim"], c["conv"]
    T = sum(new)
    C = 2 * G * D + H * E
    cols = st["proj"].split(mod.split_sizes(), -1)
    if c["channel"]:
        b, a, gate = cols[3], st["a"], st["gate"]
    else:
        gate, b, a = cols[3], cols[4], cols[5]
    (x,) = _padded(c, st["proj"][:, :C])
    tail = _first_state(c, st, mod.conv_state)
    full = torch.cat([tail, x], 1)
    y = torch.nn.functional.silu((full.unfold(1, taps, 1) * w["conv_weight"].to(F64)).sum(-1))
    ends = torch.stack([full[i, n:n + taps - 1] for i, n in enumerate(new)])
    L = y.shape[1]
    q, k = (y[..., s:s + G * D].view(B, L, G, D) for s in (0, G * D))
    v = y[..., 2 * G * D:].view(B, L, H, E)
    q, k = (z * torch.rsqrt(z.pow(2).sum(-1, keepdim=True) + 1e-6) for z in (q, k))
    q, k = (q * D ** -0.5).repeat_interleave(H // G, 2), k.repeat_interleave(H // G, 2)
    bp, ap = _padded(c, b, a)
    beta = torch.sigmoid(bp)
    g = torch.exp(-torch.exp(w["A_log"].to(F64))[:, None] *
                  torch.nn.functional.softplus(ap + w["dt_bias"].to(F64)).view(B, L, H, -1))
    S, o = _first_state(c, st, mod.state), torch.zeros(B, L, H, E, dtype=F64, device=DEV)
    for t in range(L):
        N = S * g[:, t, :, :, None]
        u = beta[:, t, :, None] * (v[:, t] - torch.matmul(k[:, t, :, None], N)[:, :, 0])
        N = N + k[:, t, :, :, None] * u[:, :, None]
        o[:, t] = torch.matmul(q[:, t, :, None], N)[:, :, 0]
        S = torch.where(_live(c, t).view(-1, 1, 1, 1), N, S)
    z = _rms(_rows_of(c, o)) * w["norm_weight"].to(F64) * torch.nn.functional.silu(gate.to(F64)).view(T, H, E)
    return dict(y=z.view(T, H * E), state=_to_slots(st, S, mod.state), conv=_to_slots(st, ends, mod.conv_state))


def _exact_scan(c, st):
    new, _ = _layout(c)
    B, H, D, E, w, T = len(new), c["heads"], c["dim"], c["vdim"], st["w"], sum(new)
    if c["rule"] == "wkv":
        q, k, v, dec = _padded(c, st["r"], st["k"], st["v"], st["w_raw"])
        L, S0, gate = q.shape[1], st["state"], st["gate"]
        dec = torch.exp(-torch.exp(dec + w["w_bias"].to(F64))).view(B, L, H, D)
        bonus = w["bonus"].to(F64)
    else:
        mod = st["mod"]
        cols = st["proj"].split(mod.split_sizes(), -1)
        gate, S0 = cols[3], mod.state
        q, k, v = _padded(c, *cols[:3])
        L = q.shape[1]
        q, k, v = q.view(B, L, H, D) * D ** -0.5, k.view(B, L, H, D), v.view(B, L, H, E)
        if c["rule"] == "gla":
            (a,) = _padded(c, st["decay_raw"])
            dec = torch.exp(torch.nn.functional.logsigmoid(a + w["decay_bias"].to(F64)) / 16.0).view(B, L, H, D)
        else:
            ig, fg = _padded(c, cols[4], cols[5])
            ig = 15.0 * torch.tanh((ig + w["i_bias"].to(F64)) / 15.0)
            fg = torch.nn.functional.logsigmoid(15.0 * torch.tanh((fg + w["f_bias"].to(F64)) / 15.0))
            n, top = _first_state(c, st, mod.norm_state[:, :, 0]), _first_state(c, st, mod.max_state[:, :, 0])
    S, o = _first_state(c, st, S0), torch.zeros(B, L, H, E, dtype=F64, device=DEV)
    for t in range(L):
        kv = k[:, t, :, :, None] * v[:, t, :, None]
        live = _live(c, t).view(-1, 1, 1, 1)
        if c["rule"] == "mlstm":
            m2 = torch.maximum(fg[:, t] + top, ig[:, t])
            f, i = torch.exp(fg[:, t] + top - m2), torch.exp(ig[:, t] - m2)
            N = f[..., None, None] * S + i[..., None, None] * kv
            n2 = f[..., None] * n + i[..., None] * k[:, t]
            den = torch.maximum((n2 * q[:, t]).sum(-1).abs(), torch.exp(-m2)) + 1e-6
            o[:, t] = torch.matmul(q[:, t, :, None], N)[:, :, 0] / den[..., None]
            n, top = torch.where(live[..., 0], n2, n), torch.where(live[..., 0, 0], m2, top)
        else:
            N = dec[:, t, :, :, None] * S + kv
            read = S + bonus[..., None] * kv if c["rule"] == "wkv" else N
            o[:, t] = torch.matmul(q[:, t, :, None], read)[:, :, 0]
        S = torch.where(live, N, S)
    act = torch.sigmoid if c["rule"] == "mlstm" else torch.nn.functional.silu
    z = _rms(_rows_of(c, o)) * w["norm_weight"].to(F64).view(-1, E) * act(gate.to(F64)).view(T, H, E)
    out = dict(y=z.view(T, H * E), state=_to_slots(st, S, S0))
    if c["rule"] == "mlstm":
        Z = mod.norm_state.shape[2]
        out["norm"] = _to_slots(st, n[:, :, None].expand(-1, -1, Z, -1), mod.norm_state)
        out["top"] = _to_slots(st, top[:, :, None].expand(-1, -1, Z), mod.max_state)
    return out


def _exact_request(c, m):
    """The dense decoder over whole sequences (its layer norms' weights are ones)."""
    lens = _lengths(dict(c, ragged=True), c["prompts"], c["length"])
    V, W, H, G, D, I = (DENSE[x] for x in ("vocab_size", "hidden_size", "num_heads", "num_kv_heads", "head_dim",
                                           "intermediate_size"))
    prompts = [[m.r.randrange(V) for _ in range(n)] for n in lens]
    given = [[m.r.randrange(V) for _ in range(c["steps"])] for _ in lens]

    def weight(name, *shape):
        return _dense_weight(name, shape).to(F64)

    embed = weight("model.embed_tokens.weight", V, W)
    xs = [embed[torch.tensor(p + g, device=DEV)] for p, g in zip(prompts, given)]
    for i in range(DENSE["num_layers"]):
        at = "model.layers.%d." % i
        qkv, o = weight(at + "self_attn.qkv_proj.weight", (H + 2 * G) * D, W), weight(at + "self_attn.o_proj.weight", W, H * D)
        qn, kn = weight(at + "self_attn.q_norm.weight", D), weight(at + "self_attn.k_norm.weight", D)
        gu, dn = weight(at + "mlp.gate_up_proj.weight", 2 * I, W), weight(at + "mlp.down_proj.weight", W, I)
        for j, x in enumerate(xs):
            T = x.shape[0]
            pos = torch.arange(T, device=DEV)
            p = _rms(x) @ qkv.t()
            q = _half_turn(_rms(p[:, :H * D].view(T, H, D)) * qn, pos, D, 1e6)
            k = _half_turn(_rms(p[:, H * D:(H + G) * D].view(T, G, D)) * kn, pos, D, 1e6)
            x = x + _attend(q, k, p[:, (H + G) * D:].view(T, G, D), D ** -0.5, 0).reshape(T, H * D) @ o.t()
            g, u = (_rms(x) @ gu.t()).split(I, -1)
            xs[j] = x + (torch.nn.functional.silu(g) * u) @ dn.t()
    norm, head = weight("model.norm.weight", W), weight("lm_head.weight", V, W)
    last = torch.stack([x[n - 1:] for x, n in zip(xs, lens)], 1)               # [steps + 1, prompts, W]
    return (_rms(last) * norm) @ head.t()


_EXACT = dict(decode=_exact_decode, prefill=_exact_prefill, attention=_exact_attention, latent=_exact_latent,
              delta=_exact_delta, scan=_exact_scan)


# ------------------------------------------------------------------ work and tolerance
def _seen(c, n, s):
    """(query, key) pairs of n queries at positions s .. s + n - 1; keys that any of them sees."""
    window, keep, chunk = c.get("window", 0), c.get("keep_first", 0), c.get("chunk", 0)
    pairs, oldest = 0, s + n
    for i in range(s, s + n):
        lo = max(0, i - window + 1) if window else 0
        if chunk:
            lo = max(lo, i // chunk * chunk)
        pairs += i + 1 - lo + min(keep, lo)
        oldest = min(oldest, lo)
    return pairs, s + n - oldest + min(keep, oldest)


def work(c):
    if c["kind"] == "request":
        lens = _lengths(dict(c, ragged=True), c["prompts"], c["length"])
        V, W, H, G, D, I, L = (DENSE[x] for x in ("vocab_size", "hidden_size", "num_heads", "num_kv_heads", "head_dim",
                                                  "intermediate_size", "num_layers"))
        per = L * ((H + 2 * G) * D * W + H * D * W + 3 * I * W)
        n, asked = c["prompts"], c["prompts"] * (c["steps"] + 1)
        pairs = sum(_seen(c, k + c["steps"], 0)[0] for k in lens)
        kv = sum(k + c["steps"] for k in lens) * 2 * G * D * 2 * L
        return dict(bytes=(c["steps"] + 1) * (per + V * W) * 2 + kv * (1 + c["steps"]) + asked * V * 4,
                    flops=2 * per * (sum(lens) + n * c["steps"]) + 2 * V * W * asked + 4 * pairs * H * D * L)
    e = 4 if c["dtype"] == "fp32" else 2
    new, past = _layout(c)
    T, H = sum(new), c["heads"]
    if c["kind"] in ("decode", "prefill", "attention", "latent"):
        seen = [_seen(c, n, s) for n, s in zip(new, past)]
        pairs, keys = sum(p for p, _ in seen), sum(k for _, k in seen)
    if c["kind"] in ("decode", "prefill"):
        ec = 1 if c.get("fp8") else e
        return dict(bytes=2 * T * H * c["dim"] * e + keys * 2 * c["kv_heads"] * c["dim"] * ec,
                    flops=4 * pairs * H * c["dim"])
    if c["kind"] == "attention":
        return dict(bytes=(T * H * (c["dim"] + c["vdim"]) + keys * c["kv_heads"] * (c["dim"] + c["vdim"])) * e,
                    flops=2 * pairs * H * (c["dim"] + c["vdim"]))
    if c["kind"] == "latent":
        D, P, R, E = c["dim"], c["rot"], c["rank"], c["vdim"]
        # the keys and values may be formed or not: whichever takes fewer operations
        formed = 2 * pairs * H * (D + P + E) + 2 * sum(n + s for n, s in zip(new, past)) * H * R * (D + E)
        absorbed = 2 * pairs * H * (2 * R + P) + 2 * T * H * R * (D + E)
        return dict(bytes=(T * H * (D + P + E) + 2 * T * (R + P) + keys * (R + P) + H * R * (D + E)) * e,
                    flops=min(formed, absorbed))
    D, E, B = c["dim"], c["vdim"], len(new)
    state = B * H * D * E * 4 * (1 + any(past))
    if c["kind"] == "delta":
        G = c["kv_heads"]
        rows = T * (2 * G * D + 3 * H * E + (H * D + H if c["channel"] else 2 * H)) * e
        return dict(bytes=rows + state, flops=T * H * D * E * 7 + T * (2 * G * D + H * E) * 2 * c["conv"])
    rows = T * H * (2 * D + 3 * E + (2 if c["rule"] == "mlstm" else D)) * e
    return dict(bytes=rows + state, flops=T * H * D * E * 5)


def tolerance(c):
    """About four times what lies between ``run`` and ``exact``."""
    if c["kind"] == "request":            # bfloat16 activations through eight layers
        return {"rel": 6e-2}
    if c["kind"] == "latent":             # two further products in bfloat16 around the attention
        return {"rel": 1.6e-2}
    return {"rel": {"fp32": 1e-5, "fp16": 1e-3, "bf16": 8e-3}[c["dtype"]]}
