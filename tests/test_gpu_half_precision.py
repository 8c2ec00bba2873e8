"""Half-precision activations through the packed arithmetic of the 16-bit kernels, against the CPU restatement of the
reference's torch oracle, where that arithmetic can go wrong: subnormal values and results, sums and products that
overflow, NaNs, and every row form of the norm kernel.

No tolerance on values: each row (head) is bit-identical to the oracle at an rstd within 3 (2) fp32 ULPs, the freedom
that the order of its sum of squares leaves."""
import pytest
import torch

from gpuk_amd import workloads
from tests.test_gpu_norm_quant import run_capi
from tests.test_gpu_rope import check_inplace, run_inplace
from tests.util import assert_bits_equal, assert_norm_rows_explained

pytestmark = pytest.mark.gpu


# (tokens, hidden): one, two, four (gated, one round) and eight chunks per lane, rows that fill their lanes and not
@pytest.mark.parametrize("tokens,hidden", [(12, 520), (12, 8192), (1100, 7168), (1300, 5128), (12, 40960)])
@pytest.mark.parametrize("quant", [0, 1, 3])
def test_norm_quant_extremes(device, tokens, hidden, quant):
    print(f"case fp16 extremes {tokens}x{hidden} q{quant}", flush=True)
    inp = workloads.norm_quant_inputs(tokens, hidden, seed=tokens + hidden, res_sigma=2.0, outlier_frac=0.01, dtype=torch.float16)
    x, r = inp.x, inp.residual
    x[0], r[0] = x[0] * 2.0 ** -20, r[0] * 2.0 ** -21       # subnormal sums
    x[1] = x[1] * 2.0 ** (torch.arange(hidden) % 24 - 14)    # every magnitude in one row
    x[2, ::7], r[2, ::7] = 60000.0, 60000.0                  # sums that overflow
    x[3, hidden - 1] = float("nan")
    x[4], r[4] = 0.0, 0.0
    x[5], r[5] = 30000.0, 30000.0                            # the largest finite row
    inp.gamma[::5] = inp.gamma[::5] * 2.0 ** -18             # subnormal products
    static = torch.tensor([0.01]) if quant == 3 else None
    assert_norm_rows_explained(inp, quant, run_capi(inp, quant, device, static_scale=static), static)


@pytest.mark.parametrize("neox", [True, False])
@pytest.mark.parametrize("head_size", [64, 128, 256])
def test_rope_small_and_large_products(device, neox, head_size):
    """Weights and table values whose products are subnormal, tiny next to their partner, or as large as the type holds."""
    print(f"case fp16 rope D={head_size} neox={neox}", flush=True)
    inp = workloads.rope_inputs(37, 13, 3, 2, head_size, seed=head_size, max_pos=64, dtype=torch.float16, is_neox=neox, random_table=True)
    inp.qkv[::3] = inp.qkv[::3] * 2.0 ** -16
    inp.cos_sin[1::4] = inp.cos_sin[1::4] * 2.0 ** -14
    inp.cos_sin[2::4, ::3] = inp.cos_sin[2::4, ::3] * 2.0 ** -11
    inp.cos_sin[3::4] = inp.cos_sin[3::4] * 2.0 ** 9
    inp.qw[::5] = inp.qw[::5] * 2.0 ** -12
    before = inp.qkv.clone()
    got = run_inplace(inp, device)
    check_inplace(inp, got, f"[fp16 D={head_size} neox={neox}]")
    assert_bits_equal(inp.qkv, before, "inputs of the oracle")
