"""Norm-quant rows that do not start on 128-byte lines, whose lanes stand at the line boundary before the row where the
workgroup has lanes to spare (16 chunks, 8 chunks, none), at one, two, four and eight chunks per lane, gated and not, run as
two launches, and in buffers that start inside a line themselves: the oracle's bits at an rstd within 3 fp32 ULPs, and
nothing written before or behind the outputs."""
import pytest
import torch

from gpuk_amd import workloads
from tests.util import assert_norm_rows_explained, canonical

pytestmark = pytest.mark.gpu


def inside(t, lead, device, fill):
    """t's shape and type in the middle of a larger buffer, `lead` elements from its (aligned) start."""
    buf = torch.full((lead + t.numel() + 64,), fill, device=device).to(t.dtype)
    return buf, buf[lead:lead + t.numel()].view(t.shape)


# hidden: 110, 119 and 125 chunks of 16-bit elements on 128 places; 129 and 401 (one chunk per lane, at the row in bfloat16 and
# fp32, at the line where 1201 rows gate their stores; two for large batches);
# 1125 (two, gated at 700 rows; four, gated, at 1257); 5121 (eight)
@pytest.mark.parametrize("tokens,hidden", [(5, 880), (37, 952), (37, 1000), (300, 1032), (1201, 1032), (3000, 1032), (2100, 3208), (700, 9000),
                                           (1257, 9000), (1500, 9000), (3, 40968)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("quant", [0, 1, 3])
def test_rows_inside_lines(device, tokens, hidden, dtype, quant):
    from gpuk_amd import capi

    if dtype == torch.float32 and hidden > 16384:
        pytest.skip("fp32 rows of this length are swept by another kernel")
    print(f"case unaligned {tokens}x{hidden} {dtype} q{quant}", flush=True)
    inp = workloads.norm_quant_inputs(tokens, hidden, seed=tokens + hidden, res_sigma=2.0, outlier_frac=0.01, dtype=dtype)
    lead = 16 // inp.x.element_size() * (tokens % 3)          # 0, 16 or 32 bytes into a line
    x, r = (inside(t, lead, device, 0.0)[1].copy_(t) for t in (inp.x, inp.residual))
    res_buf, res = inside(inp.x, lead, device, 3.0)
    norm_dtype = dtype if quant == 0 else torch.float8_e4m3fn
    norm_buf, norm = inside(torch.empty(tokens, hidden, dtype=norm_dtype), 16 * (tokens % 3), device, 3.0)
    static = torch.tensor([0.013]) if quant == 3 else None
    scale = None if quant == 0 else torch.full((tokens, 1), -1.0, device=device) if quant == 1 else static.to(device)
    g = inp.gamma.to(device)
    try:
        capi.set_tuning("norm_quant_launches", 2 if tokens == 1500 else 0)
        capi.add_rmsnorm_quant(x, r, g, res, norm, scale, inp.eps, quant)
        torch.cuda.synchronize()
    finally:
        capi.set_tuning("norm_quant_launches", 0)
    for buf, out in ((res_buf, res), (norm_buf, norm)):
        out_at = out.storage_offset()
        rest = canonical(torch.cat([buf[:out_at].float(), buf[out_at + out.numel():].float()]))
        assert bool((rest == rest[0]).all()) and float(buf[-1].float()) == 3.0, "written outside the output"
    assert_norm_rows_explained(inp, quant, (res, norm, scale), static)
