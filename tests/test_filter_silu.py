"""silu of the delta rule's filter, written out (csrc/hybrid/hybrid_delta.hip): every range of its argument against 64 bits and, bit by
bit, against the expression in fp32, in each of the kernels that have it."""
import pytest
import torch

pytestmark = pytest.mark.gpu
H, E = 2, 64
HEADS = {2: (1, 8), 1: (2, 12), 0: (1, 8)}                # form -> key heads, their size
# form, taps: rows in whole runs of eight, channels in runs with heads that are none, a channel per thread
FORMS = [(2, 2), (2, 3), (2, 4), (1, 2), (1, 3), (1, 4), (0, 2), (0, 4), (0, 5)]


def filtered(z, form, taps, dtype=torch.float32):
    """silu(z) for z [T, H * E] by the kernel ``form``: a filter whose last tap is 1, the others -0 as its bias, so that a first row's -0
    stays one."""
    from minivllm_amd.ops import hip_hybrid as hk
    G, D = HEADS[form]
    T, C = z.shape[0], 2 * G * D + H * E
    proj = torch.zeros(T, C + 2 * H + (-(C + 2 * H) % 8 if form else 1), dtype=dtype, device="cuda")
    proj[:, 2 * G * D:C] = z
    w = torch.full((C, taps), -0.0, device="cuda")
    w[:, -1] = 1
    i32 = dict(dtype=torch.int32, device="cuda")
    q, k, v, b, a = proj[:, :C + 2 * H].split([G * D, G * D, H * E, H, H], dim=-1)
    state = torch.zeros(1, taps - 1, C, device="cuda")
    qn, kn, vv, _, _ = hk.delta_prepare(
        q.view(T, G, D), k.view(T, G, D), v.view(T, H, E), b, a, w, torch.zeros(H, device="cuda"), torch.zeros(H, device="cuda"), state,
        torch.tensor([0, T], **i32), torch.arange(T, **i32), torch.zeros(1, **i32), torch.zeros(T, **i32),
        conv_bias=torch.full((C,), -0.0, device="cuda"))
    assert hk._prep_form(proj.data_ptr(), proj.stride(0), w.data_ptr(), state.data_ptr(), qn.data_ptr(), kn.data_ptr(), vv.data_ptr(),
                         taps, H, G, D, E) == form
    return vv.view(T, H * E).cpu()


def near(y, z):
    """The exponential unit's ulp and a rounding ahead of it, a sum and a quotient: below 3 of 2^-24 (with expf and an IEEE
    division 2.98 over 10^6 values)."""
    want = z.double() * torch.sigmoid(z.double())
    return ((y.double() - want).abs() <= 3 * 2.0 ** -24 * want.abs()).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form,taps", FORMS)
@pytest.mark.parametrize("reach", [1.0, 20.0, 86.0])
def test_values(reach, form, taps, dtype):
    g = torch.Generator().manual_seed(int(reach))
    z = ((torch.rand(40, H * E, generator=g) * 2 - 1) * reach).to(dtype).float()
    assert near(filtered(z.cuda(), form, taps, dtype), z)


@pytest.mark.parametrize("form,taps", FORMS)
def test_small_results(form, taps):
    """Arguments from -87 to where expf ends: their silu, down to 2.6e-37, are normal numbers as near to 64 bits as any other."""
    z = -torch.linspace(87.0, 88.72, 64 * H * E).view(64, -1)
    assert near(filtered(z.cuda(), form, taps), z)


@pytest.mark.parametrize("form,taps", FORMS)
def test_ends(form, taps):
    """Infinities, NaN, signed zeros, the smallest and largest numbers, and arguments whose exponential leaves fp32's range.  (One row: a
    filter's zero taps would make NaN of them in the rows behind.)"""
    inf, nan = float("inf"), float("nan")
    z = torch.tensor([inf, -inf, nan, 0.0, -0.0, -88.73, -104.0, -3e38, 88.0, 104.0, 1e38, 3.4e38, 1e-40, -1e-40, 2.0 ** -126, -2.0 ** -149])
    y = filtered(z.repeat(1, H * E // 16).cuda(), form, taps)[0].view(-1, 16)
    assert (y == y[0]).logical_or(y.isnan()).all()
    y = y[0]
    assert y[0] == inf and y[1].isnan() and y[2].isnan()
    assert not y[3:8].any() and y[3:8].signbit().tolist() == [False, True, True, True, True]
    assert near(y[8:12], z[8:12])
    assert ((y[12:].double() - z[12:].double() / 2).abs() <= 2.0 ** -150).all()          # half of it, rounded to a number there is
    assert (y[12:].signbit() == z[12:].signbit()).all()


# where log2(e)'s lower part, rounded instead of cut to 24 bits, puts the exponential one place off expf
PLACES = [-87.6323853, -79.0445404, -76.9907761, -74.7452698, -73.0642929, -61.6797829, -60.720314, -57.0911827, -54.5741081, -46.1522217,
          -40.9672012, -30.360157, -29.5498428, -19.8694191, -15.3136673, -7.82923794]


@pytest.mark.parametrize("form,taps", FORMS)
def test_bits(form, taps):
    """Bit by bit z / (1 + expf(-z)), as torch has it in fp32: one of every 8191 arguments from the lowest to the highest, all from -89 to
    -87, and those above.  (All 2^32 were compared once, in a program that calls both functions.)"""
    bits = torch.arange(0, 1 << 32, 8191, dtype=torch.int64)
    z = torch.cat([(bits - (bits >> 31 << 32)).to(torch.int32).view(torch.float32), torch.tensor(PLACES),
                   -(87.0 + torch.arange(1 << 18) * 2.0 ** -17)])
    z = z[z.isfinite()]
    z = torch.cat([z, z.new_zeros(-z.numel() % (H * E))]).view(-1, H * E).cuda()
    y, want = filtered(z, form, taps), (z / (1 + torch.exp(-z))).cpu()
    differ = (y.view(torch.int32) != want.view(torch.int32)) & ~((y == 0) & (z.cpu() == 0))    # (behind a first row 0 comes of -0)
    assert not differ.any(), z.cpu()[differ]
