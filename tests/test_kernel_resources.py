"""The built kernels' own metadata (no GPU needed): forms that hold their data in registers must not spill any of it to
scratch memory."""
import os
import re
import struct

import msgpack

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpuk_amd", "lib", "libgpuk_amd.so")
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    """The device ELF images in a host library: bundles of (offset, size, target) entries."""
    at = data.find(BUNDLE)
    while at >= 0:
        pos = at + len(BUNDLE) + 8
        for _ in range(struct.unpack_from("<Q", data, at + len(BUNDLE))[0]):
            offset, size, name_len = struct.unpack_from("<QQQ", data, pos)
            if b"gfx950" in data[pos + 24:pos + 24 + name_len]:
                yield data[at + offset:at + offset + size]
            pos += 24 + name_len
        at = data.find(BUNDLE, at + 1)


def kernels(elf):
    """amdhsa.kernels of the code object's metadata note (owner "AMDGPU", type 32: msgpack)."""
    table, = struct.unpack_from("<Q", elf, 0x28)
    entry, count = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, table + i * entry + 4)
        offset, size = struct.unpack_from("<QQ", elf, table + i * entry + 24)
        end = offset + size
        while kind == 7 and offset < end:   # SHT_NOTE
            name_size, desc_size, note = struct.unpack_from("<III", elf, offset)
            desc = offset + 12 + (name_size + 3) // 4 * 4
            if note == 32:
                yield from msgpack.unpackb(elf[desc:desc + desc_size], strict_map_key=False)["amdhsa.kernels"]
            offset = desc + (desc_size + 3) // 4 * 4


def test_no_scratch_where_rows_stay_in_registers():
    found = {k[".name"]: k for elf in code_objects(open(LIB, "rb").read()) for k in kernels(elf)}
    assert len(found) > 100
    # (rows of 8 chunks per lane are left out: filled bf16 ones spill a dozen registers around their reductions)
    bounded = [n for n in found if "rope_rms" in n or ("add_rmsnorm_quant" in n and "Li8E" not in n)]
    assert sum("rope_rms_token_kernel" in n for n in bounded) >= 24
    # (half precision in place with two tokens per wave: up to 24 bytes per lane, cheaper there than what avoids them)
    in_place_two = re.compile(r"rope_rms_token_kernelINS_4FP16ELi128ELb[01]ELi4ELb0ELb0ELi[13]ELb1E")
    spilled = {n: found[n][".private_segment_fixed_size"] for n in bounded}
    spilled = {n: b for n, b in spilled.items() if b > (24 if in_place_two.search(n) else 0)}
    assert not spilled, spilled


def test_gated_waves_are_all_resident():
    """The store gate of the rope kernel with one wave per group of heads counts on eight waves per SIMD (512 registers per lane)."""
    found = {k[".name"]: k[".vgpr_count"] for elf in code_objects(open(LIB, "rb").read()) for k in kernels(elf)}
    gated = {n: v for n, v in found.items() if re.search(r"rope_rms_kernelINS_4\w{4}ELi\d+ELb\dELi\dELb\dELb\dELb1E", n)}
    assert len(gated) >= 50
    assert not {n: v for n, v in gated.items() if v > 64}


def test_every_token_form_is_one_that_a_call_can_reach():
    """The rope kernel with one wave per token, in place: beyond whole tokens only rotation by halves and three or four units, two
    items per wave in half precision only."""
    names = [k[".name"] for elf in code_objects(open(LIB, "rb").read()) for k in kernels(elf) if "rope_rms_token_kernelI" in k[".name"]]
    forms = [re.search(r"INS_4(\w{4})ELi(\d+)ELb(\d)ELi(\d)ELb(\d)ELb(\d)ELi(\d)ELb(\d)ELb(\d)E", n).groups() for n in names]
    assert len(forms) == len(set(forms)) >= 200
    for dtype, _, neox, units, set_kv, _, _, two, parts in forms:
        assert set_kv == "1" or parts == "0" or (neox == "1" and units != "5" and (two == "0" or dtype == "FP16"))


def test_small_calls_pass_few_arguments():
    """The kernels that small calls launch take at most four parameters, and at most 112 bytes of them (128 and 136 with
    three position axes and a cache, or two token streams): what a launch costs the host goes by both."""
    found = {k[".name"]: k for elf in code_objects(open(LIB, "rb").read()) for k in kernels(elf)}
    seen = 0
    for name, k in found.items():
        if not re.search(r"add_rmsnorm_quant_(f32_)?rowsI|rope_rms_kernelI|rope_rms_2way_kernelI", name):
            continue
        seen += 1
        assert len([a for a in k[".args"] if not a[".value_kind"].startswith("hidden")]) <= 4, name
        head = re.search(r"rope_rms_kernelINS_4[BF][FP]16ELi(64|128|256)ELb[01]ELi([13])ELb([01])ELb([01])ELb([01])E", name)
        most = 128 if "2way" in name else 112
        if head:   # (the gate of launches that fill half the chip comes on top)
            most += 8 * int(head[5]) + (8 * int(head[4]) + {64: 8, 128: 16, 256: 32}[int(head[1])] if head[2] == "3" else 0)
        assert k[".kernarg_segment_size"] <= most, (name, k[".kernarg_segment_size"])
    assert seen > 250
