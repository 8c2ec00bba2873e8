"""The functional operator behind GPUKDistEnv.allreduce_add_rms_fused: its meta kernels without a GPU; on the GPU the same
outputs as the in-place operator, what it refuses, and that neither autograd nor functional transforms see more than they
did through the in-place one."""
import pytest
import torch

import gpuk_amd
from gpuk_amd import workloads
from tests.util import assert_bits_equal


@pytest.mark.parametrize("quant,dtype", [(0, torch.bfloat16), (1, torch.float8_e4m3fn)])
def test_meta_shapes(quant, dtype):
    x = torch.empty(5, 3, 64, dtype=torch.bfloat16, device="meta")
    res, norm, scale = torch.ops.gpuk.add_rms_fused(x, x, x[0, 0], 1e-6, quant)
    assert (res.shape, res.dtype, norm.shape, norm.dtype) == (x.shape, x.dtype, x.shape, dtype)
    assert scale.dtype == torch.float32 and tuple(scale.shape) == ((5, 1) if quant else (1,))
    res, norm = torch.ops.gpuk.add_rms_fused.static(x, x, x[0, 0], 1e-6, torch.empty(1, device="meta"))
    assert (res.dtype, norm.shape, norm.dtype) == (x.dtype, x.shape, torch.float8_e4m3fn)


@pytest.mark.parametrize("quant", [2, 3, 7, -1])
@pytest.mark.parametrize("where", ["meta", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_modes_without_a_scale_to_return(where, quant):
    """The scale is an output here: a static scale has its own overload, and unknown modes are refused on meta tensors too."""
    x = torch.zeros(2, 64, dtype=torch.bfloat16, device=where)
    with pytest.raises(RuntimeError, match="add_rms_fused.static"):
        torch.ops.gpuk.add_rms_fused(x, x, x[0], 1e-6, quant)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["none", "dynamic", "static"])
def test_equals_the_in_place_operator(device, mode):
    inp = workloads.norm_quant_inputs(7, 1032, seed=7, res_sigma=2.0)
    x, r, g = inp.x.to(device), inp.residual.to(device), inp.gamma.to(device).requires_grad_()
    env = gpuk_amd.GPUKDistEnv(device_id=device.index or 0)
    static = torch.full((1, 1), 0.02, device=device) if mode == "static" else None
    res, norm, scale = env.allreduce_add_rms_fused(x, r, g, inp.eps, fp8_out=mode != "none", static_scale=static)
    assert not res.requires_grad and res.grad_fn is None and norm.grad_fn is None   # weights may be parameters
    quant = {"none": 0, "dynamic": 1, "static": 3}[mode]
    want_res, want_norm = torch.empty_like(r), torch.empty_like(x, dtype=norm.dtype)
    want_scale = static.reshape(1) if static is not None else torch.empty(7, 1, device=device)
    gpuk_amd.allreduce_rms(0, x, r, g, want_res, want_norm, want_scale, inp.eps, quant)
    torch.cuda.synchronize()
    assert_bits_equal(res, want_res.cpu(), "residual_out")
    assert_bits_equal(norm.view(torch.uint8), want_norm.view(torch.uint8).cpu(), "norm_out")
    if mode != "none":
        assert torch.equal(scale, want_scale)
    if static is not None:
        assert scale.data_ptr() == static.data_ptr() and scale.shape == (1,)


@pytest.mark.gpu
def test_refusals(device):
    env = gpuk_amd.GPUKDistEnv(device_id=device.index or 0)
    x = torch.zeros(4, 64, dtype=torch.bfloat16, device=device)
    g = torch.ones(64, dtype=torch.bfloat16, device=device)
    for bad in ((x.t(), x, g), (x, x.t(), g), (x, x[:2], g), (x, x.half(), g), (x, x, g[:32]), (x[:, :60].contiguous(), x, g),
                (x, x.cpu(), g), (x.cpu(), x, g), (x.int(), x.int(), g.int())):
        with pytest.raises(RuntimeError):
            env.allreduce_add_rms_fused(*bad, 1e-6, fp8_out=True)
    with pytest.raises(NotImplementedError):
        env.allreduce_add_rms_fused(x.cpu(), x.cpu(), g.cpu(), 1e-6)
    for bad in (torch.ones(2, device=device), torch.ones(1), torch.ones(1, device=device).double()):
        with pytest.raises(ValueError):
            env.allreduce_add_rms_fused(x, x, g, 1e-6, fp8_out=True, static_scale=bad)
    for scale in (None, torch.ones(1, device=device)):
        with pytest.raises(RuntimeError, match="Batching rule"):
            torch.func.vmap(lambda a: env.allreduce_add_rms_fused(a, a, g, 1e-6, fp8_out=True, static_scale=scale)[0])(x[None])
    res, norm, scale = env.allreduce_add_rms_fused(x[:0], x[:0], g, 1e-6, fp8_out=True)   # an empty batch
    assert res.shape == (0, 64) and norm.dtype == torch.float8_e4m3fn and scale.shape == (0, 1)
