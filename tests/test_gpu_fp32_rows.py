"""fp32 rows of the norm kernel, which share the 16-bit kernel's arrangement: every form of a row (one, two, four chunks per
lane; lanes filled or not), the store gate, batches run as two launches, runs of rows per XCD, and values where its short
quotients could go wrong.

No tolerance on values: each row is bit-identical to the oracle at an rstd within 3 fp32 ULPs, the freedom that the order
of its sum of squares leaves."""
import pytest
import torch

from gpuk_amd import workloads
from tests.util import assert_norm_rows_explained, canonical

pytestmark = pytest.mark.gpu


def run(inp, quant, device, static=None, alias=False):
    from gpuk_amd import capi

    x, r, g = inp.x.to(device), inp.residual.to(device), inp.gamma.to(device)
    res = r if alias else torch.empty_like(x)
    tokens, hidden = x.shape
    norm = torch.full((tokens + 1, hidden), 3.0, device=device)   # one row more than the call may write
    norm = norm if quant == 0 else norm.to(torch.float8_e4m3fn)
    guard = canonical(norm[-1])
    scale = None if quant == 0 else torch.full((tokens, 1), -1.0, device=device) if quant == 1 else static.to(device)
    capi.add_rmsnorm_quant(x, r, g, res, norm, scale, inp.eps, quant)
    torch.cuda.synchronize()
    assert torch.equal(canonical(norm[-1]), guard), "written behind the last row"
    return res, norm[:-1], scale


# one chunk per lane; two, filled and not, one row and gated; four, filled and not, gated (one round); two launches of half
# the rows; more than a round, in runs of 64 rows per XCD with rows left over
@pytest.mark.parametrize("tokens,hidden", [(3, 264), (1, 4096), (300, 4096), (900, 1032), (1100, 4096), (1300, 2568), (5, 16384),
                                           (2400, 4096), (4200, 4096)])
@pytest.mark.parametrize("quant", [0, 1, 3])
def test_row_forms(device, tokens, hidden, quant):
    print(f"case fp32 rows {tokens}x{hidden} q{quant}", flush=True)
    inp = workloads.norm_quant_inputs(tokens, hidden, seed=tokens + hidden, res_sigma=2.0, outlier_frac=0.01, dtype=torch.float32)
    static = torch.tensor([0.013]) if quant == 3 else None
    assert_norm_rows_explained(inp, quant, run(inp, quant, device, static, alias=tokens == 1100), static)


@pytest.mark.parametrize("quant,static", [(0, None), (1, None), (3, 0.01), (3, 1e-17), (3, 1e-30)])
@pytest.mark.parametrize("tokens,hidden", [(16, 264), (16, 7168), (700, 4104)])
def test_extreme_values(device, tokens, hidden, quant, static):
    """Zero rows, NaNs, infinities, sums of squares that overflow, subnormal elements next to ordinary ones, weights so large
    that a quotient by the static scale overflows, and scales too small for a reciprocal."""
    print(f"case fp32 extremes {tokens}x{hidden} q{quant} {static}", flush=True)
    inp = workloads.norm_quant_inputs(tokens, hidden, seed=hidden, res_sigma=1.0, dtype=torch.float32)
    x, r = inp.x, inp.residual
    x[0], r[0] = 0.0, 0.0
    x[1, 5] = float("nan")
    x[2, 7] = float("inf")
    x[3] = x[3] * 1e30
    x[4], r[4] = x[4] * 2.0 ** -75, r[4] * 2.0 ** -76      # squares underflow: rstd from eps alone
    x[5, ::2], r[5, ::2] = x[5, ::2] * 1e-38, r[5, ::2] * 1e-39
    x[6], r[6] = x[6] * 2.0 ** (torch.arange(hidden) % 60 - 50).float(), 0.0
    x[7], r[7] = -x[7].abs() * 1e-20, 0.0
    inp.gamma[::9] = inp.gamma[::9] * 1e25 if static == 1e-17 else inp.gamma[::9] * 1e-12
    inp.gamma[4] = -inp.gamma[4]
    s = None if static is None else torch.tensor([static])
    assert_norm_rows_explained(inp, quant, run(inp, quant, device, s), s)


@pytest.mark.parametrize("threads,nchunk", [(0, 8), (512, 8), (1024, 8), (1024, 2), (1024, 1), (448, 4), (0, 1)])
def test_forced_shapes(device, threads, nchunk):
    """The tuning keys choose another launch, never another result; eight chunks per lane, which only the 16-bit kernel has,
    become four."""
    from gpuk_amd import capi

    print(f"case fp32 forced threads={threads} nchunk={nchunk}", flush=True)
    capi.set_tuning("norm_quant_nchunk", nchunk)
    capi.set_tuning("norm_quant_threads", threads)
    try:
        for tokens, hidden in ((301, 4096), (301, 1032), (37, 16384)):
            inp = workloads.norm_quant_inputs(tokens, hidden, seed=threads + hidden, res_sigma=2.0, outlier_frac=0.01, dtype=torch.float32)
            for quant in (0, 1, 3):
                static = torch.tensor([0.013]) if quant == 3 else None
                assert_norm_rows_explained(inp, quant, run(inp, quant, device, static), static)
    finally:
        capi.set_tuning("norm_quant_nchunk", 0)
        capi.set_tuning("norm_quant_threads", 0)


# one, two and four chunks per lane, lanes filled and not: weights asked for once the row has landed (below 7168 elements), once
# rstd is known (from there), and at once (two waves; two chunks on four and one row per compute unit; without codes up to 32 long
# rows, and rows of two chunks that do not fill their lanes; more than a round); gated rows of one chunk per lane on nine and eleven
# waves, which without codes ask once landed as well
@pytest.mark.parametrize("tokens,hidden", [(5, 3320), (3, 1536), (33, 5120), (200, 2568), (6, 10240), (6, 10248), (3, 3840), (7, 3624), (7, 2424),
                                           (9, 8192), (9, 7176), (4, 16384), (4, 15000), (40, 1024), (700, 5640), (450, 2304), (400, 2568), (5, 4104), (300, 1536), (33, 8192), (33, 7176), (33, 16384), (33, 15000), (300, 1456)])
@pytest.mark.parametrize("quant", [0, 1, 3])
def test_weight_orders(device, tokens, hidden, quant):
    print(f"case fp32 weights {tokens}x{hidden} q{quant}", flush=True)
    inp = workloads.norm_quant_inputs(tokens, hidden, seed=tokens + hidden, res_sigma=2.0, outlier_frac=0.01, dtype=torch.float32)
    static = torch.tensor([0.013]) if quant == 3 else None
    assert_norm_rows_explained(inp, quant, run(inp, quant, device, static, alias=tokens == 9), static)
