"""Dynamic quantisation to maxima other than 448 and 240.  The quotient of a row's largest element by its scale exceeds the
maximum by one ULP in up to one row in seventeen; where the maximum lies halfway between two codes (400, 336, 100) that ULP
would turn into the next code, beyond the maximum, and the oracle's clamp keeps it.  Every form of a row against the
oracle's bits at an rstd within 3 fp32 ULPs."""
import pytest
import torch

from gpuk_amd import workloads
from tests.test_gpu_norm_quant import run_capi
from tests.util import assert_norm_rows_explained

pytestmark = pytest.mark.gpu


# rows of one, two, four (gated) and eight chunks per lane, and swept; 301 is no such maximum
@pytest.mark.parametrize("tokens,hidden", [(600, 264), (600, 1024), (1300, 5128), (40, 24576), (40, 90112)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("fp8_max", [400.0, 336.0, 100.0, 301.0])
def test_dynamic_scale_at_other_maxima(device, tokens, hidden, dtype, fp8_max):
    print(f"case fp8_max {fp8_max} {tokens}x{hidden} {dtype}", flush=True)
    inp = workloads.norm_quant_inputs(tokens, hidden, seed=tokens + hidden, res_sigma=2.0, outlier_frac=0.01, dtype=dtype)
    got = run_capi(inp, 1, device, fp8_max=fp8_max)
    assert_norm_rows_explained(inp, 1, got, fp8_max=fp8_max)
    assert float(got[1].float().abs().max()) <= fp8_max
