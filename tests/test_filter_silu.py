"""silu of the delta rule's filter, written out (csrc/hybrid/hybrid_delta.hip): every range of its argument against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
G, D, H, E = 1, 8, 2, 64


def filtered(z, taps, fast):
    """silu(z) for z [T, H * E]: a filter whose last tap is 1 and whose others are 0.  ``fast``: rows in whole runs of eight."""
    from minivllm_amd.ops import hip_hybrid as hk
    T, C = z.shape[0], 2 * G * D + H * E
    proj = torch.zeros(T, C + 2 * H + (8 - 2 * H % 8 if fast else 1), device="cuda")
    proj[:, 2 * G * D:C] = z
    w = torch.zeros(C, taps, device="cuda")
    w[:, -1] = 1
    i32 = dict(dtype=torch.int32, device="cuda")
    q, k, v, b, a = proj[:, :C + 2 * H].split([G * D, G * D, H * E, H, H], dim=-1)
    vv = hk.delta_prepare(q.view(T, G, D), k.view(T, G, D), v.view(T, H, E), b, a, w, torch.zeros(H, device="cuda"),
                          torch.zeros(H, device="cuda"), torch.zeros(1, taps - 1, C, device="cuda"), torch.tensor([0, T], **i32),
                          torch.arange(T, **i32), torch.zeros(1, **i32), torch.zeros(T, **i32))[2]
    return vv.view(T, H * E).cpu()


@pytest.mark.parametrize("taps,fast", [(4, True), (4, False), (2, True), (5, False)])
@pytest.mark.parametrize("reach", [1.0, 20.0, 86.0])
def test_values(reach, taps, fast):
    """The exponential unit's ulp and a rounding ahead of it, a sum and a quotient: below 3 of 2^-24 (with expf and an IEEE
    division 2.98 over 10^6 values)."""
    g = torch.Generator().manual_seed(int(reach))
    z = (torch.rand(40, H * E, generator=g) * 2 - 1) * reach
    y, want = filtered(z.cuda(), taps, fast).double(), z.double() * torch.sigmoid(z.double())
    assert ((y - want).abs() <= 3 * 2.0 ** -24 * want.abs()).all()


@pytest.mark.parametrize("fast", [True, False])
def test_ends(fast):
    """Infinities, NaN, signed zeros, and arguments whose exponential leaves fp32's range.  (One row: a filter's zero taps
    would make NaN of them in the rows behind.)"""
    inf, nan = float("inf"), float("nan")
    z = torch.tensor([inf, -inf, nan, 0.0, 88.0, 104.0, 1e38, -88.0, -104.0, -200.0, -1e38, 1e-40, -1e-40, 1.0, -1.0, 2.0])
    y = filtered(z.repeat(1, H * E // 16).cuda(), 2, fast)[0].view(-1, 16)
    assert (y[:, 0] == inf).all() and y[:, 1].isnan().all() and y[:, 2].isnan().all()
    rest = z[3:].double()
    assert torch.allclose(y[:, 3:].double(), (rest / (1 + torch.exp(-rest))).expand(y.shape[0], -1), rtol=3 * 2.0 ** -24, atol=1e-36)


@pytest.mark.parametrize("fast", [True, False])
def test_small_results(fast):
    """Arguments from -87 to where expf ends: their silu, down to 2.6e-37, are normal numbers as near to 64 bits as any other."""
    z = -torch.linspace(87.0, 88.72, 64 * H * E).view(64, -1)
    y, want = filtered(z.cuda(), 4, fast).double(), z.double() * torch.sigmoid(z.double())
    assert ((y - want).abs() <= 3 * 2.0 ** -24 * want.abs()).all()


# where log2(e)'s lower part, rounded instead of cut to 24 bits, puts the exponential one place off expf
PLACES = [-87.6323853, -79.0445404, -76.9907761, -74.7452698, -73.0642929, -61.6797829, -60.720314, -57.0911827, -54.5741081, -46.1522217,
          -40.9672012, -30.360157, -29.5498428, -19.8694191, -15.3136673, -7.82923794]


@pytest.mark.parametrize("taps,fast", [(4, True), (4, False), (3, True), (5, False)])
def test_bits(taps, fast):
    """Bit by bit z / (1 + expf(-z)), as torch has it in fp32: one of every 8191 arguments from the lowest to the highest, all from -89 to
    -87, and those above.  (All 2^32 were compared once, in a program that calls both functions.)"""
    bits = torch.arange(0, 1 << 32, 8191, dtype=torch.int64)
    z = torch.cat([(bits - (bits >> 31 << 32)).to(torch.int32).view(torch.float32), torch.tensor(PLACES),
                   -(87.0 + torch.arange(1 << 18) * 2.0 ** -17)])
    z = z[z.isfinite()]
    z = torch.cat([z, z.new_zeros(-z.numel() % (H * E))]).view(-1, H * E).cuda()
    y, want = filtered(z, taps, fast), (z / (1 + torch.exp(-z))).cpu()
    differ = (y.view(torch.int32) != want.view(torch.int32)) & ~((y == 0) & (z.cpu() == 0))    # (the filter's sum makes 0 of -0)
    assert not differ.any(), z.cpu()[differ]
