"""The one-wave-per-token rope kernel on tokens split into parts: forced onto small batches, the bits of the kernel with one wave
per group of heads and the oracle's, with a 16-bit cache and in place, one item per wave and two."""
import pytest
import torch

from gpuk_amd import capi
from tests.test_gpu_rope import check_inplace, check_set_kv, make, run_inplace, run_set_kv

pytestmark = pytest.mark.gpu

CASES = [
    # tokens, (hq, hk, hv), head size, neox, sections (None: one axis), interleaved, two items, fp16
    (61, (16, 2, 2), 128, True, None, False, False, False),      # one part of three units, the last a quarter full
    (62, (12, 12, 12), 128, True, None, False, False, False),    # three V chunks per lane
    (45, (40, 8, 8), 128, True, None, False, False, False),      # two parts of three
    (33, (40, 8, 8), 128, False, None, False, False, True),
    (29, (64, 8, 8), 128, True, None, False, False, False),      # three parts of three
    (41, (48, 8, 8), 128, False, None, False, False, False),     # two parts of four, the last unit idle
    (37, (28, 4, 4), 256, True, None, False, False, False),      # two parts of four
    (23, (32, 8, 8), 256, False, None, False, False, True),      # two parts of five
    (19, (17, 0, 1), 256, True, None, False, False, False),      # a part whose last unit holds one head, no K heads, one V head
    (31, (0, 41, 3), 128, True, None, False, False, False),      # no Q heads, two parts, the second nearly all idle lanes
    (50, (28, 4, 4), 128, True, [24, 20, 20], True, False, False),   # merged table rows, one part
    (50, (28, 4, 4), 128, False, [24, 20, 20], False, False, True),
    (27, (40, 8, 8), 128, True, [24, 20, 20], True, False, False),
    (26, (28, 4, 4), 256, False, [48, 40, 40], True, False, False),
    (61, (16, 2, 2), 128, True, None, False, True, False),       # two items of three units, an odd count
    (45, (40, 8, 8), 128, True, None, False, True, True),
    (30, (40, 8, 8), 128, False, [24, 20, 20], True, True, False),   # the two items of a wave lie in different tokens
    (29, (28, 4, 4), 256, True, None, False, True, True),
    (40, (28, 4, 4), 128, True, [16, 24, 24], True, True, False),
    (1, (40, 8, 8), 128, True, None, False, True, False),        # one token: its two parts are the two items of one wave
]


# (in place there are no forms of five units but for whole tokens of one table row, nor of two items in bfloat16, nor, which the query
# does not know, with pairwise rotation or merged table rows of those)
IN_PLACE = {7: 0, 8: 0, 14: 0, 16: 0, 19: 0}


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("gate", [-1, 600])
def test_tokens_in_parts(device, case, gate):
    tokens, heads, D, neox, sections, interleaved, two, fp16 = CASES[case]
    print(f"case parts {CASES[case]} gate={gate}", flush=True)
    inp = make(tokens, heads[0], D, neox, seed=700 + case, mrope=sections is not None, interleaved=interleaved, hk=heads[1], hv=heads[2])
    if sections is not None:
        inp.mrope_section = sections
        inp.positions[:, ::3] = inp.positions[:1, ::3]    # text tokens among the others: three equal positions
    if fp16:
        inp.qkv, inp.qw, inp.kw, inp.cos_sin = (t.to(torch.float16) for t in (inp.qkv, inp.qw, inp.kw, inp.cos_sin))
        inp.kv_dtype = torch.float16
    if tokens > 2:
        inp.kv_loc[1], inp.kv_loc[tokens - 1] = -1, -5
    axes = 3 if sections else 1
    try:
        capi.set_tuning("rope_token_waves", 1)
        base, base_inplace = run_set_kv(inp, device), run_inplace(inp, device)
        capi.set_tuning("rope_token_waves", 3 if two else 2)
        capi.set_tuning("rope_token_gate", gate)
        assert capi.rope_rms_launch_shape(tokens, *heads, D, axes, inp.qkv.dtype, True, False)[3] == (2 if two else 1), "the case must reach the kernel under test"
        assert capi.rope_rms_launch_shape(tokens, *heads, D, axes, inp.qkv.dtype, False, False)[3] == IN_PLACE.get(case, 2 if two else 1)
        got, got_inplace = run_set_kv(inp, device), run_inplace(inp, device)
    finally:
        capi.set_tuning("rope_token_waves", 0)
        capi.set_tuning("rope_token_gate", -1)
    raw = lambda t: t.cpu().contiguous().view(torch.uint8)
    for name, a, b in zip(("q_out", "k_cache", "v_cache"), got[:3], base[:3]):
        assert torch.equal(raw(a), raw(b)), f"{name}: the two kernels differ"
    assert torch.equal(raw(got_inplace), raw(base_inplace)), "in place: the two kernels differ"
    check_set_kv(inp, got, f"[parts {case}]")
    check_inplace(inp, got_inplace, f"[parts {case}, in place]")


@pytest.mark.parametrize("tokens,heads,D,waves", [(1536, (40, 8, 8), 128, 3072), (2048, (40, 8, 8), 128, 4096), (2304, (40, 8, 8), 128, 4096),
                                                  (4096, (40, 8, 8), 128, 4096), (1365, (64, 8, 8), 128, 4095), (2048, (28, 4, 4), 256, 4096), (4096, (28, 4, 4), 256, 4096)])
def test_parts_by_rule(device, tokens, heads, D, waves):
    """The sizes the rule takes, at the edges of what a round holds: every item taken exactly once."""
    print(f"case parts by rule {tokens} {heads} {D}", flush=True)
    inp = make(tokens, heads[0], D, True, seed=tokens, hk=heads[1], hv=heads[2])
    inp.kv_loc[5::11] = -1
    assert capi.rope_rms_launch_shape(tokens, *heads, D, 1, inp.qkv.dtype, True, False)[:2] == ((waves + 3) // 4, 256)
    got = run_set_kv(inp, device)
    try:
        capi.set_tuning("rope_token_waves", 1)
        base = run_set_kv(inp, device)
    finally:
        capi.set_tuning("rope_token_waves", 0)
    for name, a, b in zip(("q_out", "k_cache", "v_cache"), got[:3], base[:3]):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16)), f"{name}: the two kernels differ"


@pytest.mark.parametrize("tokens,heads,D,neox,sections,fp16", [
    (2731, (16, 2, 2), 128, True, None, False), (2390, (12, 12, 12), 128, False, None, True), (4097, (16, 2, 2), 128, True, [24, 20, 20], True),
    (1792, (28, 4, 4), 128, False, [16, 24, 24], True), (4097, (28, 4, 4), 128, True, [24, 20, 20], True), (1152, (24, 8, 8), 256, True, None, False),
    (2179, (14, 2, 2), 256, False, None, False), (1844, (32, 8, 8), 128, False, None, False), (1537, (48, 8, 8), 128, True, [24, 20, 20], False)])
def test_choice_changes_no_bits(device, tokens, heads, D, neox, sections, fp16):
    """Calls at the lines of the rule, as it chooses and with one wave per group of heads: the same bits, with a cache and in
    place, for either rotation, table rows that are merged and tokens without a slot."""
    print(f"case choice {tokens} {heads} {D} neox={neox} {sections} fp16={fp16}", flush=True)
    inp = make(tokens, heads[0], D, neox, seed=tokens, mrope=sections is not None, interleaved=sections is not None and sections[0] == 24, hk=heads[1], hv=heads[2])
    if sections is not None:
        inp.mrope_section = sections
        inp.positions[:, ::3] = inp.positions[:1, ::3]
    if fp16:
        inp.qkv, inp.qw, inp.kw, inp.cos_sin = (t.to(torch.float16) for t in (inp.qkv, inp.qw, inp.kw, inp.cos_sin))
        inp.kv_dtype = torch.float16
    inp.kv_loc[3::13] = -1
    got = [*run_set_kv(inp, device)[:3], run_inplace(inp, device)]
    try:
        capi.set_tuning("rope_token_waves", 1)
        base = [*run_set_kv(inp, device)[:3], run_inplace(inp, device)]
    finally:
        capi.set_tuning("rope_token_waves", 0)
    for name, a, b in zip(("q_out", "k_cache", "v_cache", "in place"), got, base):
        assert torch.equal(a.cpu().contiguous().view(torch.uint8), b.cpu().contiguous().view(torch.uint8)), f"{name}: the two kernels differ"


@pytest.mark.parametrize("tokens,heads,D,neox,fp8,fp16", [
    (615, (32, 8, 8), 128, True, False, True), (615, (32, 8, 8), 128, False, False, True), (456, (64, 8, 8), 128, True, True, True), (1707, (32, 8, 8), 64, True, False, False),
    (2177, (28, 4, 4), 64, False, False, False), (257, (64, 64, 64), 128, True, True, False), (1639, (8, 1, 1), 256, True, False, True)])
def test_gate_and_workgroup_change_no_bits(device, tokens, heads, D, neox, fp8, fp16):
    """Calls at the lines of the rule for the gate, the lines and the workgroup of the kernel with one wave per group of heads,
    as it chooses and without a gate in single waves that store through the L2: the same bits, with a cache and in place."""
    print(f"case gate rule {tokens} {heads} {D} neox={neox} fp8={fp8} fp16={fp16}", flush=True)
    inp = make(tokens, heads[0], D, neox, seed=tokens + D, fp8=fp8, hk=heads[1], hv=heads[2])
    if fp16:
        inp.qkv, inp.qw, inp.kw, inp.cos_sin = (t.to(torch.float16) for t in (inp.qkv, inp.qw, inp.kw, inp.cos_sin))
        if not fp8:
            inp.kv_dtype = torch.float16
    inp.kv_loc[3::13] = -1
    got = [*run_set_kv(inp, device)[:3], run_inplace(inp, device)]
    plain = {"rope_token_waves": (1, 0), "rope_unit_gate": (0, -1), "rope_stream_rows": (1, 0), "rope_block_threads": (64, 0)}
    try:
        for key, (value, _) in plain.items():
            capi.set_tuning(key, value)
        base = [*run_set_kv(inp, device)[:3], run_inplace(inp, device)]
    finally:
        for key, (_, rule) in plain.items():
            capi.set_tuning(key, rule)
    for name, a, b in zip(("q_out", "k_cache", "v_cache", "in place"), got, base):
        assert torch.equal(a.cpu().contiguous().view(torch.uint8), b.cpu().contiguous().view(torch.uint8)), f"{name}: the launches differ"
