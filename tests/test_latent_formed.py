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
