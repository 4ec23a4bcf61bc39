"""Rotation and store of latent rows by a wave per token, against the plain PyTorch form."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from minivllm_amd.ops import hip_hybrid as hk
from minivllm_amd.ops import torch_seqmix as ref


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,H,D,P,R,dims,neighbours,shift", [
    # sizes of one pass and of several, a part that is not rotated, tokens that do not fill a workgroup, both
    # orders of pairs; last: rows that start off 16 bytes, and dims that pairs of runs do not fill
    (4097, 16, 128, 64, 512, 64, False, 0), (4099, 3, 8, 24, 520, 16, False, 0), (4098, 20, 64, 64, 8, 64, True, 0),
    (4096, 2, 24, 32, 1048, 8, True, 0), (7, 16, 128, 64, 512, 64, False, 0), (1025, 65, 8, 24, 512, 16, False, 0),
    (1021, 65, 8, 24, 512, 16, True, 0), (4100, 2, 16, 16, 64, 16, False, 4), (4100, 2, 16, 16, 64, 8, False, 0)])
@pytest.mark.parametrize("own_values", [False, True])
def test_turn_store(dt, T, H, D, P, R, dims, neighbours, shift, own_values):
    torch.manual_seed(T + R)
    q_all, dkv_all = torch.randn(T, H * (D + P) + 8).to(dt), torch.randn(T, R + P + 16).to(dt)
    part = lambda x, y: (x[:, shift:shift + H * (D + P)].view(T, H, D + P), y[:, shift:shift + R + P])  # noqa: E731
    (q, dkv), (gq, gdkv) = part(q_all, dkv_all), part(q_all.cuda(), dkv_all.cuda())
    w, inv = torch.rand(R) + 0.5, torch.rand(dims // 2)
    pos = torch.randint(0, 3000, (T,), dtype=torch.int32)
    slots = torch.randperm(T + 64)[:T].to(torch.int32)
    slots[5::7] = -1                                                 # rows that store nothing
    k = torch.randn(T + 64, 1, 1, R + P).to(dt)
    v = torch.randn(T + 64, 1, 1, R).to(dt) if own_values else None
    q_abs = torch.zeros(H, T, R, dtype=dt)
    gk, gv = k.cuda(), None if v is None else v.cuda()
    out = hk.latent_rope_store(q_abs.cuda(), gq, gdkv, w.cuda(), 1e-6, pos.cuda(), inv.cuda(), dims, gk, gv, slots.cuda(),
                               neighbours, 1.25, False)
    want = ref.latent_rope_store(q_abs, q, dkv, w, 1e-6, pos, inv, dims, k, v, slots, neighbours, 1.25, False)
    # float: the angle reaches 3000, so its fp32 rounding 2^-24 * 3000 = 2e-4 turns entries below 6 * 1.25; both
    # sides round it alike, what is left is sine, cosine and sums.  bfloat16: half a unit of 8 bits either side
    tol = dict(rtol=2 ** -7, atol=2 ** -7) if dt == torch.bfloat16 else dict(rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(out.cpu(), want, **tol)
    torch.testing.assert_close(gk.cpu(), k, **tol)
    if own_values:
        torch.testing.assert_close(gv.cpu(), v, **tol)
