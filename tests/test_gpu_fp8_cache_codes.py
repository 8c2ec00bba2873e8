"""Every 16-bit pattern through an fp8 cache: V rows carry no arithmetic but the quantisation, so their codes are the converter's
on all 65,536 values, at scales whose quotients are ordinary, clamped, tiny and out of the short form's range.  Which form of the
conversion takes a value is chosen for a wave's 512 values at once: every form gets all the values that it accepts."""
import pytest
import torch

from gpuk_amd import capi

pytestmark = pytest.mark.gpu

D, HV = 128, 8                     # a token's V row is two passes of a wave, 512 values each
PASS = 512


def check(rows, scale, dtype, device):
    """rows [tokens, HV * D]: their codes against the quotient, rounded, clamped and converted by torch."""
    T = rows.shape[0]
    qkv = torch.zeros(T, 2 + HV, D, dtype=dtype)
    qkv[:, 2:] = rows.reshape(T, HV, D)
    w, table = torch.ones(D, dtype=dtype), torch.ones(4, D, dtype=dtype)
    d = lambda t: t.to(device)
    kc = torch.zeros(T, 1, D, dtype=torch.float8_e4m3fn, device=device)
    vc = torch.zeros(T, HV, D, dtype=torch.float8_e4m3fn, device=device)
    q = torch.empty(T, 1, D, dtype=dtype, device=device)
    capi.rope_rms_set_kv(d(qkv), d(w), d(w), d(table), torch.zeros(T, dtype=torch.int64, device=device), T, 1, 1, HV, D, True, 1e-6,
                         q, kc, vc, torch.arange(T, device=device), 1.0, scale, None, False)
    torch.cuda.synchronize()
    quotient = (rows.float() / torch.tensor(scale, dtype=torch.float32)).to(dtype).float()
    want = torch.where(quotient.isnan(), quotient, quotient.clamp(-448.0, 448.0)).to(torch.float8_e4m3fn)
    got, nan = vc.cpu().view(torch.uint8).reshape(T, -1), quotient.isnan()
    assert torch.equal(got[~nan], want.view(torch.uint8)[~nan])
    assert bool(((got[nan] & 0x7f) == 0x7f).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("scale", [1.0, 0.02, 0.05, 1.5, 2.0, 1 / 3, 1.0 - 2.0 ** -24, 240.0, 1e-4, 3.0 ** 37, 3.0 ** -37, 3.0 ** 40, 2.0 ** -62])
def test_every_value(device, dtype, scale):
    print(f"case fp8 codes {dtype} scale={scale}", flush=True)
    ordered = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype)
    mixed = ordered[torch.randperm(65536, generator=torch.Generator().manual_seed(3))]
    for values in (mixed, ordered):   # an infinity or a NaN in every pass, and in order
        check(values.reshape(-1, HV * D), scale, dtype, device)


def magnitudes(largest_quotient, s):
    """All bfloat16 patterns of both signs whose quotient by s is at most this, in mixed order, zeros filling up the last row."""
    patterns = torch.arange(0x7f80, dtype=torch.int32)
    quotients = patterns.to(torch.int16).view(torch.bfloat16).double() / s.double()
    top = int((quotients <= largest_quotient).sum()) - 1
    bits = torch.cat([torch.arange(top + 1), torch.arange(top + 1) + 0x8000])
    bits = bits[torch.randperm(len(bits), generator=torch.Generator().manual_seed(5))]
    rows = torch.zeros(-(-len(bits) // (HV * D)) * HV * D, dtype=torch.int64)
    rows[:len(bits)] = bits
    return rows.to(torch.int16).view(torch.bfloat16).reshape(-1, HV * D), top


@pytest.mark.parametrize("scale", [1.0, 0.02, 0.05, 1.5, 2.0, 1 / 3, 1.0 - 2.0 ** -24, 240.0, 1e-4, 3.0 ** 37, 3.0 ** -37, 2.0 ** -60, 2.0 ** 60])
def test_every_form_of_the_conversion(device, scale):
    print(f"case fp8 forms scale={scale}", flush=True)
    s = torch.tensor(scale, dtype=torch.float32)
    unclamped, top = magnitudes(448.0, s)
    largest = float(unclamped.double().abs().max() / s.double())
    assert 444.0 < largest <= 448.0                       # up to the largest code's value: the next pattern has to be clamped
    check(unclamped, scale, torch.bfloat16, device)
    finite, finite_top = magnitudes(2.0 ** 60, s)        # quotients of any size, clamped
    check(finite, scale, torch.bfloat16, device)
    # passes of values up to it but for one, in every lane's first or last place in turn
    bits = unclamped.reshape(-1).view(torch.int16).to(torch.int32)[:PASS] & 0xffff
    above = int((480.0 * s).view(torch.int32)) >> 16       # would not be the top code unless clamped
    offenders = [top, top + 1, top + 0x8001, above, above + 0x8000, finite_top, finite_top + 1, 0x7f7f, 0xff7f, 0x7f80, 0xff80, 0x7f81, 0xffc0, 0x7fff]
    passes = []
    for i, value in enumerate(offenders):
        for place in (0, 1, 6, 7, PASS - 8, PASS - 1, 8 * (7 * i % 64) + i % 8):
            one = bits.clone()
            one[place] = value & 0xffff
            passes.append(one)
    passes += [bits] * (len(passes) % 2)
    check(torch.cat(passes).to(torch.int16).view(torch.bfloat16).reshape(-1, HV * D), scale, torch.bfloat16, device)
