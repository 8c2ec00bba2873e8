"""Every 16-bit pattern through an fp8 cache: V rows carry no arithmetic but the quantisation, so their codes are the converter's
on all 65,536 values, at scales whose quotients are ordinary, clamped, tiny and out of the short form's range."""
import pytest
import torch

from gpuk_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("scale", [1.0, 0.02, 0.05, 1.5, 2.0, 1 / 3, 240.0, 1e-4, 3.0 ** 37, 3.0 ** -37, 3.0 ** 40, 2.0 ** -62])
def test_every_value(device, dtype, scale):
    print(f"case fp8 codes {dtype} scale={scale}", flush=True)
    T, D, hv = 64, 128, 8                                 # 64 rows of 1024 values
    v = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype).reshape(T, hv, D)
    v = v.flatten()[torch.randperm(65536, generator=torch.Generator().manual_seed(3))].reshape(T, hv, D)
    ordered = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype).reshape(T, hv, D)
    for rows in (v, ordered):                             # mixed, every wave with something to clamp, and in order
        qkv = torch.zeros(T, 2 + hv, D, dtype=dtype)
        qkv[:, 2:] = rows
        w, table = torch.ones(D, dtype=dtype), torch.ones(4, D, dtype=dtype)
        d = lambda t: t.to(device)
        kc = torch.zeros(T, 1, D, dtype=torch.float8_e4m3fn, device=device)
        vc = torch.zeros(T, hv, D, dtype=torch.float8_e4m3fn, device=device)
        q = torch.empty(T, 1, D, dtype=dtype, device=device)
        capi.rope_rms_set_kv(d(qkv), d(w), d(w), d(table), torch.zeros(T, dtype=torch.int64, device=device), T, 1, 1, hv, D, True, 1e-6,
                             q, kc, vc, torch.arange(T, device=device), 1.0, scale, None, False)
        torch.cuda.synchronize()
        quotient = (rows.float() / torch.tensor(scale, dtype=torch.float32)).to(dtype).float()
        want = torch.where(quotient.isnan(), quotient, quotient.clamp(-448.0, 448.0)).to(torch.float8_e4m3fn)
        got, nan = vc.cpu().view(torch.uint8), quotient.isnan()
        assert torch.equal(got[~nan], want.view(torch.uint8)[~nan])
        assert bool(((got[nan] & 0x7f) == 0x7f).all())
