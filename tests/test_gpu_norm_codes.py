"""GPU: fp8 codes over every significand a normed value and a row's maximum can have.  The kernels take the quotient by a
reciprocal in two parts, which is the IEEE quotient up to the code it rounds to; here against the IEEE quotient."""
import pytest
import torch

pytestmark = pytest.mark.gpu

BINADES = 19   # from the row's maximum down to values whose code is zero


@pytest.mark.parametrize("dtype,bits,step", [(torch.bfloat16, 8, 1), (torch.float16, 11, 16)])
@pytest.mark.parametrize("fp8_max", [448.0, 240.0, 300.0])
def test_codes_of_every_significand(device, dtype, bits, step, fp8_max):
    print(f"case codes {dtype} fp8_max={fp8_max}", flush=True)
    from gpuk_amd import capi

    one = 1 << (bits - 1)
    grid = torch.cat([(one + torch.arange(one)).double() / (2 * one) * 2.0 ** -k for k in range(BINADES)])
    grid[1::2] *= -1
    hidden = grid.numel()
    gamma = torch.ones(hidden, dtype=dtype, device=device)
    for top in range(one, 2 * one, step):
        amax = top / (2 * one)
        row = torch.where(grid.abs() <= amax, grid, torch.zeros_like(grid)).to(dtype)
        row[0] = amax
        eps = 1.0 - row.double().square().mean().item()   # rstd is 1 but for the order of the sum: the normed row is the row
        x = row.reshape(1, hidden).to(device)
        out = torch.empty_like(x)
        codes = torch.empty(1, hidden, dtype=torch.float8_e4m3fn, device=device)
        scale = torch.empty(1, 1, device=device)
        normed = torch.empty_like(x)
        capi.add_rmsnorm_quant(x, torch.zeros_like(x), gamma, out, normed, None, eps, 0)
        capi.add_rmsnorm_quant(x, torch.zeros_like(x), gamma, out, codes, scale, eps, 1, fp8_max)
        assert torch.equal(normed.cpu().flatten().float(), row.float()), top
        want_scale = torch.tensor(amax) / fp8_max
        assert scale.item() == want_scale.item(), top
        want = (row.float() / want_scale).clamp(-fp8_max, fp8_max).to(torch.float8_e4m3fn)
        got = codes.cpu().flatten().view(torch.uint8)
        assert torch.equal(got, want.view(torch.uint8)), (top, int((got != want.view(torch.uint8)).sum()))


# (1 - 2^-24: a significand of ones, which the short form leaves to the division; 2^-61 and 2^61: beyond its range)
@pytest.mark.parametrize("scale", [0.05, 0.0123, 1.0, 1 / 3, 1.0 - 2.0 ** -24, 2.0 ** -61, 2.0 ** 61, float("nan")])
@pytest.mark.parametrize("dtype,bits", [(torch.bfloat16, 8), (torch.float16, 11)])
def test_codes_with_a_static_scale(device, dtype, bits, scale):
    print(f"case static codes {dtype} scale={scale}", flush=True)
    from gpuk_amd import capi

    one = 1 << (bits - 1)
    grid = torch.cat([(one + torch.arange(one)).double() / one * 2.0 ** k for k in range(-14, 8)])
    grid[1::2] *= -1
    row = torch.cat([grid, torch.zeros(8, dtype=torch.double)]).to(dtype)
    hidden = row.numel()
    # a weight per element and a row of ones: the normed row is the weights, whatever they are
    gamma = row.clone()
    gamma[-8:] = torch.tensor([0.0, -0.0, float("inf"), -float("inf"), float("nan"), 1.0, -1.0, 448.0])
    x = torch.ones(1, hidden, dtype=dtype, device=device)
    out, codes = torch.empty_like(x), torch.empty(1, hidden, dtype=torch.float8_e4m3fn, device=device)
    capi.add_rmsnorm_quant(x, torch.zeros_like(x), gamma.to(device), out, codes, torch.full((1,), scale, device=device), 0.0, 3)
    want = (gamma.float() / torch.tensor(scale)).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    got = codes.cpu().flatten().view(torch.uint8)
    nan = (want & 0x7F) == 0x7F
    assert torch.equal((got & 0x7F) == 0x7F, nan) and torch.equal(got[~nan], want[~nan])
