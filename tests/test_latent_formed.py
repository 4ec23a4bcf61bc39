"""Latent attention over prompts with keys and values formed per head: kernels, and when they are taken."""
import math

import pytest
import torch

gpu = pytest.mark.gpu


def _step(lens, qlens, bs, R, P):
    pages = [-(-n // bs) for n in lens]
    tables, at, perm = torch.zeros(len(lens), max(pages), dtype=torch.int32), 0, torch.randperm(sum(pages))
    for b, n in enumerate(pages):
        tables[b, :n] = perm[at:at + n]
        at += n
    cache = torch.randn(sum(pages), bs, 1, R + P).bfloat16()
    cu = torch.tensor([0] + torch.tensor(qlens).cumsum(0).tolist(), dtype=torch.int32)
    pos = torch.cat([torch.arange(n - m, n) for n, m in zip(lens, qlens)]).to(torch.int32)
    return tables, cache, cu, pos


@gpu
@pytest.mark.parametrize("H,D,E,R,P,bs,window,lens,qlens", [
    # all widths at once; prompts of one row, on both sides of a tile, behind a prefix, and of no rows
    (16, 128, 128, 512, 64, 256, 0, [1, 31, 32, 33, 300, 64, 700], [1, 31, 32, 33, 300, 0, 257]),
    (6, 128, 128, 256, 64, 64, 40, [97, 128, 129, 200], [97, 128, 29, 1]),
    (3, 64, 40, 128, 128, 32, 0, [160, 95, 256], [160, 64, 225]),
    (1, 8, 8, 64, 8, 32, 7, [1, 70], [1, 70]),
    (2, 104, 120, 192, 72, 96, 0, [90] * 70, [90, 1] * 35),          # more sequences than a wave has lanes
])
@pytest.mark.parametrize("with_sink", [False, True])
def test_formed_prompts(H, D, E, R, P, bs, window, lens, qlens, with_sink):
    from minivllm_amd.ops import hip_hybrid as hk
    torch.manual_seed(H + R)
    T = sum(qlens)
    tables, cache, cu, pos = _step(lens, qlens, bs, R, P)
    q, q_rot = torch.randn(T, H, D + P).bfloat16(), torch.randn(T, H, P).bfloat16()
    up_k, up_v = (torch.randn(H, D, R) * R ** -0.5).bfloat16(), (torch.randn(H, R, E) * R ** -0.5).bfloat16()
    sink, scale = (2.0 * torch.randn(H) if with_sink else None), (D + P) ** -0.5
    got = hk.latent_formed_prompts(q.cuda(), q_rot.cuda(), cache.cuda(), up_k.cuda(), up_v.cuda(), cu.cuda(), tables.cuda(),
                                   pos.cuda(), scale, None if sink is None else sink.cuda(), max(qlens), max(lens), window)
    assert got.shape == (T, H, E)
    for b, (n, m) in enumerate(zip(lens, qlens)):
        if m == 0:
            continue
        rows = cache[tables[b, :-(-n // bs)].long()].reshape(-1, R + P)[:n].double()
        sl = slice(int(cu[b]), int(cu[b + 1]))
        # keys and values as the kernel holds them, rounded to bfloat16 (a sum may round to either side: up to
        # 2^-8 of a value in few places, far below the bound's share for them)
        k = torch.einsum("nr,hdr->hnd", rows[:, :R], up_k.double()).bfloat16().double()
        v = torch.einsum("nr,hre->hne", rows[:, :R], up_v.double()).bfloat16().double()
        s = torch.einsum("mhd,hnd->hmn", q[sl, :, :D].double(), k) + torch.einsum("mhp,np->hmn", q_rot[sl].double(), rows[:, R:])
        back = pos[sl].long()[:, None] - torch.arange(n)[None]
        s = (s * scale).masked_fill((back < 0) | ((back >= window) if window else False), -math.inf)
        if with_sink:
            s = torch.cat([s, sink.double()[:, None, None].expand(H, m, 1)], -1)
        want = torch.einsum("hmn,hne->mhe", s.softmax(-1)[..., :n], v)
        # the result is rounded to bfloat16 (2^-9 of itself); a key's or value's other rounding moves single rows by less
        assert float((got[sl].cpu().double() - want).norm() / want.norm()) < 2.0 ** -8, b


@gpu
def test_infinities_and_nan_stay_in_their_rows():
    """A latent that is not finite reaches the queries that see it and no earlier ones."""
    from minivllm_amd.ops import hip_hybrid as hk
    torch.manual_seed(1)
    H, D, E, R, P, n = 4, 128, 128, 128, 64, 200
    tables, cache, cu, pos = _step([n, n], [n, n], 64, R, P)
    q, q_rot = torch.randn(2 * n, H, D + P).bfloat16().cuda(), torch.randn(2 * n, H, P).bfloat16().cuda()
    up_k, up_v = ((torch.randn(H, *s) * R ** -0.5).bfloat16().cuda() for s in ((D, R), (R, E)))

    def run(c):
        return hk.latent_formed_prompts(q, q_rot, c.cuda(), up_k, up_v, cu.cuda(), tables.cuda(), pos.cuda(), 0.07, None, n, n)
    clean = run(cache)
    bad = cache.clone()
    bad[tables[1, 100 // 64], 100 % 64, 0, 5] = float("nan")
    got = run(bad)
    # (the rows before it that share its tile are worked out key by key: another sum, the same up to a rounding of
    # the result to bfloat16 either way, 2^-8 of its size)
    assert torch.equal(got[:n + 96], clean[:n + 96]) and torch.isnan(got[n + 100:]).all()
    assert float((got[n + 96:n + 100] - clean[n + 96:n + 100]).float().norm() / clean[n + 96:n + 100].float().norm()) < 2.0 ** -8


@gpu
def test_rows_behind_too_short_a_workspace_are_left_alone():
    """A longest context that is given too short costs the rows it leaves no room for, and nothing else."""
    from minivllm_amd.ops import hip_hybrid as hk
    torch.manual_seed(2)
    H, R, P, lens = 2, 64, 8, [64, 64, 96]
    tables, cache, cu, pos = _step(lens, lens, 32, R, P)
    q, q_rot = torch.randn(sum(lens), H, 16 + P).bfloat16().cuda(), torch.randn(sum(lens), H, P).bfloat16().cuda()
    up = torch.randn(H, 16, R).bfloat16().cuda(), torch.randn(H, R, 16).bfloat16().cuda()
    a = (cache.cuda(), *up, cu.cuda(), tables.cuda(), pos.cuda(), 0.2, None, 96)
    full, short = hk.latent_formed_prompts(q, q_rot, *a, 96), hk.latent_formed_prompts(q, q_rot, *a, 64)
    assert torch.equal(full[:128], short[:128])                      # (a workgroup's rows are all there or left alone)


@gpu
@pytest.mark.parametrize("change,taken", [
    (dict(), True), (dict(dtype=torch.float32), False), (dict(max_k=0), False), (dict(max_q=65, max_k=64), False),
    (dict(max_k=128), True), (dict(max_k=161), False), (dict(bs=16), False), (dict(bs=48), False), (dict(R=96), False),
    (dict(D=136), False), (dict(D=124), False), (dict(P=136), False), (dict(E=136), False), (dict(slice_q=True), True),
    (dict(shift_q=True), False), (dict(turn_up=True), False)])
def test_when_keys_and_values_are_formed(change, taken):
    """Sizes, types, strides and alignments that the kernels have, and no more memory than the other form."""
    from minivllm_amd.ops import hip_hybrid as hk
    c = dict(dict(dtype=torch.bfloat16, D=128, E=128, R=320, P=64, bs=32, max_q=64, max_k=64, T=128, seqs=2), **change)
    H, w = 2, c["D"] + c["P"]
    z = lambda *s: torch.zeros(*s, dtype=c["dtype"], device="cuda")
    q = z(c["T"], H * w + 8)[:, :H * w].view(c["T"], H, w) if c.get("slice_q") else z(c["T"], H, w)
    if c.get("shift_q"):
        q = z(c["T"] * H * w + 4)[4:].view(c["T"], H, w)
    up_k = z(H, c["R"], c["D"]).transpose(1, 2) if c.get("turn_up") else z(H, c["D"], c["R"])
    got = hk.latent_formed_ok(q, z(c["T"], c["R"] + c["P"]), up_k, z(H, c["R"], c["E"]), z(8, c["bs"], 1, c["R"] + c["P"]),
                              torch.zeros(2, 4, dtype=torch.int32, device="cuda"), c["seqs"], c["max_q"], c["max_k"])
    assert got == taken


@pytest.mark.parametrize("R", [64, 448, 512, 576, 640, 960, 1024, 4096])
@pytest.mark.parametrize("P", [8, 64, 128])
def test_ranks_whose_weights_have_as_many_bits(R, P):
    """Formed only where the other form holds its weights in two bfloat16 parts too."""
    from minivllm_amd.ops import hip_hybrid as hk
    T, H, D = 64, 2, 128
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16)
    cache = z(2, 32, 1, R + P)
    taken = hk.latent_formed_ok(z(T, H, D + P), z(T, R + P), z(H, D, R), z(H, R, D), cache,
                                torch.zeros(1, 2, dtype=torch.int32), 1, 32, 32)
    assert taken == hk.latent_attention_ok(z(H, T, R), cache, P) == (R <= 512)


def _turned(x, pos, base=10000.0):
    """Entries i and i + n / 2 of the last dimension turn together (64 bits)."""
    n = x.shape[-1]
    a = pos.double()[:, None, None] * (base ** (-torch.arange(0, n, 2, dtype=torch.float64) / n))
    x1, x2 = x[..., :n // 2], x[..., n // 2:]
    return torch.cat([x1 * a.cos() - x2 * a.sin(), x2 * a.cos() + x1 * a.sin()], -1)


@gpu
@pytest.mark.parametrize("R,bs,formed", [(512, 32, True), (192, 64, True), (576, 32, False), (512, 16, False)])
@pytest.mark.parametrize("window,sink", [(0, False), (70, True)])
def test_steps_through_the_layer(monkeypatch, R, bs, formed, window, sink):
    """A layer's steps over one cache: prompts of several lengths, portions behind a prefix, next tokens, prompts with
    riders, a prompt behind what those wrote; rows of no sequence in between.  The steps of prompts alone run with keys
    and values formed where the rule has it, steps of few rows in one call, and are no further from 64 bits than with
    attention in the latents' coordinates, call by call."""
    from minivllm_amd import ops
    from minivllm_amd.layers.attention import LatentAttention
    from minivllm_amd.layers.rotary_embedding import HalfRotation
    from minivllm_amd.ops import hip_hybrid as hk
    from minivllm_amd.utils.context import set_context
    torch.manual_seed(R + bs)
    H, D, P, E, eps, scale, nseq, room = 4, 64, 32, 72, 1e-6, (64 + 32) ** -0.5, 3, 256
    up_k, up_v = torch.randn(H * D, R) * R ** -0.5, torch.randn(H * E, R) * R ** -0.5
    norm, weight_sink = 1 + 0.1 * torch.randn(R), torch.randn(H)
    tables = torch.randperm(nseq * room // bs).to(torch.int32).view(nseq, -1)
    layers = {}
    for form in ("rule", "absorbed"):
        a = LatentAttention(H, D, P, E, R, scale, window, HalfRotation(P, 10000.0), eps, sink=sink).cuda()
        a.latent_norm.copy_(norm)
        a.load_expansions(up_k, up_v, torch.empty(0, dtype=torch.bfloat16, device="cuda"))
        if sink:
            a.core.sink.copy_(weight_sink)
        a.core.k_cache = torch.full((tables.numel(), bs, 1, R + P), float("nan"), dtype=torch.bfloat16, device="cuda")
        a.core.v_cache = a.core.k_cache[..., :R]
        layers[form] = a
    monkeypatch.setattr(hk, "LATENT_ROWS", 100 * R)                       # (the steps lie on both sides of it)
    taken = []
    for name in ("latent_formed_prompts", "latent_rows", "latent_attention_prefill", "latent_attention_decode"):
        def spy(*args, _f=getattr(hk, name), _name=name, **kw):
            out = _f(*args, **kw)
            if out is not None or _name != "latent_rows":
                taken.append(_name)
            return out
        monkeypatch.setattr(hk, name, spy)
    rule, few = ops.latent_formed_ok, ops.latent_rows
    ku, vu = up_k.bfloat16().double().view(H, D, R), up_v.bfloat16().double().view(H, E, R)
    rows = torch.zeros(nseq, room, R + P, dtype=torch.float64)              # what the cache should hold
    past, squares = [0] * nseq, dict(rule=0.0, absorbed=0.0, of=0.0)

    def step(seqs, new, riders=0, behind=0):
        """Tokens of sequences (the first ``riders`` with one each), ``behind`` rows of none after them."""
        T = sum(new) + behind
        q, dkv = torch.randn(T, H, D + P).bfloat16(), torch.randn(T, R + P).bfloat16()
        pos = torch.tensor([past[s] + i for s, n in zip(seqs, new) for i in range(n)] + [0] * behind, dtype=torch.int32)
        owner = [b for b, n in enumerate(new) for _ in range(n)] + [-1] * behind
        slots = [int(tables[seqs[b], int(p) // bs]) * bs + int(p) % bs if b >= 0 else -1 for b, p in zip(owner, pos)]
        total = [past[s] + n for s, n in zip(seqs, new)]
        ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
        kw = dict(positions=pos.cuda(), num_seqs=len(seqs), block_tables=tables[seqs].cuda(), slot_mapping=ints(slots))
        prompts = new[riders:]
        if prompts:
            cu = lambda ns: ints([0] + torch.tensor(ns).cumsum(0).tolist())
            kw.update(is_prefill=True, cu_seqlens_q=cu(new), cu_seqlens_k=cu(total), max_seqlen_q=max(new),
                      max_seqlen_k=max(total), row_seq=ints(owner), num_decode_seqs=riders,
                      num_prefill_tokens=sum(prompts))
        if riders:
            kw.update(context_lens=ints(total[:riders]), max_context_len=max(total[:riders]))
        got, ways = {}, {}
        for form, a in layers.items():
            monkeypatch.setattr(ops, "latent_formed_ok", rule if form == "rule" else lambda *args: False)
            monkeypatch.setattr(ops, "latent_rows", few if form == "rule" else lambda *args: None)
            set_context(**kw)
            taken.clear()
            with torch.inference_mode():
                got[form] = a(q.cuda(), dkv.cuda()).double().cpu()
            ways[form] = list(taken)
        c = dkv[:, :R].double()
        c = c * torch.rsqrt(c.pow(2).mean(-1, keepdim=True) + eps) * norm.double()
        turned = torch.cat([c, _turned(dkv[:, None, R:].double(), pos)[:, 0]], -1)
        at = 0
        for s, n, m in zip(seqs, new, total):
            rows[s, past[s]:m] = turned[at:at + n]
            seen = rows[s, :m]
            k, v = (torch.einsum("nr,hdr->hnd", seen[:, :R], u) for u in (ku, vu))
            one = slice(at, at + n)
            w = torch.einsum("thd,hnd->htn", q[one, :, :D].double(), k) \
                + torch.einsum("thp,np->htn", _turned(q[one, :, D:].double(), pos[one]), seen[:, R:])
            back = pos[one].long()[:, None] - torch.arange(m)[None]
            w = (w * scale).masked_fill((back < 0) | ((back >= window) if window else False), -math.inf)
            if sink:
                w = torch.cat([w, weight_sink.double()[:, None, None].expand(H, n, 1)], -1)
            want = torch.einsum("htn,hne->the", w.softmax(-1)[..., :m], v)
            for form in got:
                # rounded to bfloat16, 2^-9 of a value each: the cached rows, the turned queries, keys or absorbed queries,
                # values or sums of latents, the result
                assert float((got[form][one] - want).norm() / want.norm()) < 5 * 2.0 ** -9, (form, s, n, m)
                squares[form] += float((got[form][one] - want).pow(2).sum()) * bool(prompts and not riders)
            past[s] = m
            at += n
        if R > 512 and behind:
            assert not got["rule"][at:].any()
        has = lambda *names: sorted(names) if R <= 512 else []
        assert sorted(ways["absorbed"]) == has(*["latent_attention_decode"] * bool(riders), *["latent_attention_prefill"] * bool(prompts))
        return sorted(ways["rule"]) if R <= 512 else ways["rule"] or None

    one_call = ["latent_rows"] if R <= 512 else None
    call_by_call = ["latent_attention_prefill"] if R <= 512 else None
    formed_or = lambda other: ["latent_formed_prompts"] if formed else other
    assert step([0, 1, 2], [5, 65, 96], behind=6) == formed_or(call_by_call)
    assert step([1, 0], [64, 75], behind=1) == formed_or(call_by_call)     # behind 65 and 5 tokens
    assert step([2, 1, 0], [1, 1, 1], riders=3) == one_call
    assert step([2, 0], [1, 40], riders=1, behind=3) == (["latent_attention_decode", "latent_attention_prefill"] if R <= 512 else None)
    assert step([0], [80]) == formed_or(one_call)
    # the two forms round the same number of times: their errors differ by chance only (a tenth allowed)
    assert squares["rule"] <= 1.21 * squares["absorbed"]
