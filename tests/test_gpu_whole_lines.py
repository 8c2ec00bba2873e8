"""Heads of 64 elements whose lines are loaded and stored whole, two heads exchanged among eight lanes (calls that stream
their stores, in place, with a 16-bit cache and two-stream): the same bits as the form that moves half lines, the oracle's bits, and nothing
written outside the Q and K heads, where heads are odd in number, units are partly filled and stores are gated."""
import pytest
import torch

from tests.test_gpu_rope import check_inplace, check_set_kv, make, run_inplace, run_set_kv
from tests.test_gpu_rope_2way import make as make_2way
from tests.util import assert_bits_equal, assert_rotated_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gate", [0, 300])
@pytest.mark.parametrize("neox,mrope", [(True, False), (False, True)])
@pytest.mark.parametrize("tokens,hq,hk,hv", [(1, 1, 0, 1), (3, 1, 1, 0), (7, 13, 4, 3), (5, 16, 17, 2), (9, 64, 64, 64)])
def test_in_place(device, tokens, hq, hk, hv, neox, mrope, gate):
    from gpuk_amd import capi

    print(f"case whole lines {tokens} tokens {hq}+{hk}+{hv} neox={neox} mrope={mrope} gate={gate}", flush=True)
    inp = make(tokens, hq, 64, neox, seed=tokens + hq, mrope=mrope, interleaved=True, hk=hk, hv=hv)
    if tokens == 5:
        inp.qkv, inp.qw, inp.kw, inp.cos_sin = (t.to(torch.float16) for t in (inp.qkv, inp.qw, inp.kw, inp.cos_sin))
    try:
        capi.set_tuning("rope_unit_gate", gate)
        capi.set_tuning("rope_stream_rows", 1)
        half = run_inplace(inp, device)
        capi.set_tuning("rope_stream_rows", 2)
        whole = run_inplace(inp, device)
    finally:
        capi.set_tuning("rope_unit_gate", -1)
        capi.set_tuning("rope_stream_rows", 0)
    assert_bits_equal(whole, half.cpu(), "whole and half lines")
    check_inplace(inp, whole, "whole lines")


@pytest.mark.parametrize("gate", [0, 300])
@pytest.mark.parametrize("neox,mrope", [(True, False), (False, True)])
@pytest.mark.parametrize("tokens,hq,hk,hv", [(1, 1, 0, 1), (5, 0, 1, 1), (7, 13, 4, 3), (9, 16, 17, 2), (11, 32, 8, 8), (9, 64, 64, 64)])
def test_with_a_cache(device, tokens, hq, hk, hv, neox, mrope, gate):
    """A lane's two pieces may belong to a Q and a K head, to heads on both sides of a unit, or to none; a token without a slot."""
    from gpuk_amd import capi

    print(f"case whole lines, cache {tokens} tokens {hq}+{hk}+{hv} neox={neox} mrope={mrope} gate={gate}", flush=True)
    inp = make(tokens, hq, 64, neox, seed=tokens + hq, mrope=mrope, interleaved=True, hk=hk, hv=hv)
    if tokens == 9:
        inp.qkv, inp.qw, inp.kw, inp.cos_sin = (t.to(torch.float16) for t in (inp.qkv, inp.qw, inp.kw, inp.cos_sin))
        inp.kv_dtype = torch.float16
    if tokens > 5:
        inp.kv_loc[2] = -1
    try:
        capi.set_tuning("rope_unit_gate", gate)
        capi.set_tuning("rope_stream_rows", 1)
        half = run_set_kv(inp, device)
        capi.set_tuning("rope_stream_rows", 2)
        whole = run_set_kv(inp, device)
    finally:
        capi.set_tuning("rope_unit_gate", -1)
        capi.set_tuning("rope_stream_rows", 0)
    for name, a, b in zip(("q_out", "k_cache", "v_cache"), whole[:3], half[:3]):
        assert_bits_equal(a, b.cpu(), f"whole and half lines: {name}")
    check_set_kv(inp, whole, "whole lines, cache")


@pytest.mark.parametrize("B,T0,T1,Hq,Hk", [(1, 1, 0, 1, 1), (2, 3, 5, 5, 3), (2, 7, 2, 16, 17)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_two_streams(device, B, T0, T1, Hq, Hk, dtype):
    from gpuk_amd import capi
    from oracle import torch_oracle as O

    D = 64
    for il in (False, True):
        c = make_2way(B, T0, T1, Hq, Hk, D, seed=T0 + 10 * Hq, dtype=dtype)
        d = lambda t: t.to(device)
        got = {}
        try:
            for policy in (1, 2):
                capi.set_tuning("rope_stream_rows", policy)
                out = [torch.full((B * (T0 + T1) + 1, h, D), 7.0, dtype=dtype, device=device) for h in (Hq, Hk)]
                capi.rope_rms_2way(d(c["q0"]), d(c["k0"]), d(c["q1"]), d(c["k1"]), *[d(w) for w in c["w"]], d(c["cs0"]),
                                   d(c["cs1"]), B, T0, T1, Hq, Hk, D, il, 1e-6, *out)
                torch.cuda.synchronize()
                got[policy] = [o.cpu() for o in out]
        finally:
            capi.set_tuning("rope_stream_rows", 0)
        ref = O.rope_rms_2way_ref(c["q0"], c["k0"], c["q1"], c["k1"], *c["w"], c["cs0"], c["cs1"], B, T0, T1, Hq, Hk, D, il, 1e-6)
        for whole, half, want in zip(got[2], got[1], ref):
            assert_bits_equal(whole, half, "whole and half lines")   # the row behind the output included
            assert_rotated_close(whole[:-1].reshape(want.shape), want, f"two streams il={il}")
