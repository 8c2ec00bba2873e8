"""CPU-only checks of the boundary: the C-ABI library loads and exports every symbol its header declares,
the torch library registers the reference's operator schemas, argument validation rejects what it must
without touching a GPU, and the host-side byte accounting matches the published per-configuration figures."""
import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "gpuk_amd.h")


def declared_functions():
    src = open(HEADER).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    return sorted(set(re.findall(r"\b(gpuk_[a-z0-9_]+)\s*\(", src)))


def test_library_exports_every_declared_symbol():
    from gpuk_amd import capi

    names = declared_functions()
    assert set(names) == set(capi.EXPORTS), (names, capi.EXPORTS)
    lib = ctypes.CDLL(os.path.join(ROOT, "gpuk_amd", "lib", "libgpuk_amd.so"))
    for n in names:
        assert getattr(lib, n) is not None
    assert capi.lib().gpuk_abi_version() == 2
    assert capi.lib().gpuk_status_string(0) == b"ok"
    assert b"unsupported" in capi.lib().gpuk_status_string(2)


def test_argument_validation_needs_no_gpu():
    """Bad arguments are rejected before any launch (status codes, not exceptions or aborts)."""
    from gpuk_amd import capi

    L = capi.lib()
    buf = ctypes.create_string_buffer(4096)
    p = ctypes.addressof(buf)
    p = (p + 15) & ~15
    f = L.gpuk_add_rmsnorm_quant
    assert f(p, p, p, p, p, p, -1, 1024, 1e-6, 0, 1, 448.0, None) == 1      # negative tokens
    assert f(p, p, p, p, p, p, 4, 1020, 1e-6, 0, 1, 448.0, None) == 2       # hidden % 8
    assert f(p, p, p, p, p, p, 4, 1024, 1e-6, 7, 1, 448.0, None) == 2       # unknown dtype
    assert f(p, p, p, p, p, p, 4, 1024, 1e-6, 0, 2, 448.0, None) == 2       # e4m3fnuz
    assert f(p, p, p, p, p, p, 4, 1024, 1e-6, 0, 9, 448.0, None) == 2       # unknown quant
    assert f(p, p, p, p, p, None, 4, 1024, 1e-6, 0, 1, 448.0, None) == 1    # dynamic quant needs scale
    assert f(p + 2, p, p, p, p, p, 4, 1024, 1e-6, 0, 1, 448.0, None) == 3   # misaligned
    assert f(p, p, p, p, p, p, 4, 1024, 1e-6, 0, 1, 0.0, None) == 1         # fp8_max must be positive
    assert f(None, None, None, None, None, None, 0, 1024, 1e-6, 0, 1, 448.0, None) == 0   # empty batch is a no-op
    sec = (ctypes.c_int64 * 3)(16, 16, 16)
    r = L.gpuk_rope_rms
    assert r(p, p, p, p, p, 0, 1, 3, 4, 2, 2, 2, 128, 1, sec, 0, 1e-6, 0, None) == 1     # sections sum to 48, not 64
    assert r(p, p, p, p, p, 0, 1, 1, 4, 2, 2, 2, 96, 1, None, 0, 1e-6, 0, None) == 2     # head size
    assert r(p, p, p, p, p, 0, 1, 2, 4, 2, 2, 2, 128, 1, None, 0, 1e-6, 0, None) == 1    # n_axes
    assert r(p, p, p, p, p, 0, 1, 3, 4, 2, 2, 2, 128, 1, None, 0, 1e-6, 0, None) == 1    # mRoPE without sections
    assert r(None, None, None, None, None, 0, 1, 1, 0, 2, 2, 2, 128, 1, None, 0, 1e-6, 0, None) == 0   # no tokens
    s = L.gpuk_rope_rms_set_kv
    assert s(p, p, p, p, p, 0, 1, 1, 4, 2, 2, 2, 128, 1, None, 0, 1e-6, 0, p, p, p, p, 1.0, 1.0, 5, None) == 2  # kv dtype
    assert s(p, p, p, p, p, 0, 1, 1, 4, 2, 2, 2, 128, 1, None, 0, 1e-6, 0, p, p, p, p, 0.0, 1.0, 1, None) == 1  # fp8 scale
    assert s(p, p, p, p, p, 0, 1, 1, 4, 2, 2, 2, 128, 1, None, 0, 1e-6, 0, None, p, p, p, 1.0, 1.0, 0, None) == 1
    w = L.gpuk_rope_rms_2way
    assert w(p, p, p, p, p, p, p, p, p, p, 1, 2, 2, 2, 2, 96, 0, 1e-6, 0, p, p, None) == 2     # head size
    assert w(p, p, p, p, p, p, p, p, p, p, 1, -2, 2, 2, 2, 128, 0, 1e-6, 0, p, p, None) == 1   # negative tokens
    assert w(p, p, p, p, p, p, p, p, p, p, 1, 2, 2, 2, 2, 128, 0, 1e-6, 0, None, p, None) == 1  # missing output
    assert w(p, p, p, p, p, p, p, p, p, p, 0, 2, 2, 2, 2, 128, 0, 1e-6, 0, p, p, None) == 0    # empty batch
    assert L.gpuk_copy_bytes(p, p, 24, None) == 1 and L.gpuk_copy_bytes(p, p, 0, None) == 0
    assert L.gpuk_read_bytes(p, 24, p, None) == 1 and L.gpuk_read_bytes(p, 0, p, None) == 0
    assert L.gpuk_read_bytes(p, 32, None, None) == 1 and L.gpuk_read_bytes(p + 4, 32, p, None) == 3
    assert L.gpuk_fill_bytes(p, 24, 1, None) == 1 and L.gpuk_fill_bytes(None, 32, 1, None) == 1
    assert L.gpuk_fill_bytes(p, 0, 1, None) == 0 and L.gpuk_fill_bytes(p + 8, 32, 1, None) == 3
    assert L.gpuk_empty_grid(4, 100, 0, None) == 1 and L.gpuk_empty_grid(4, 2048, 0, None) == 1
    assert L.gpuk_empty_grid(4, 256, 1 << 20, None) == 1 and L.gpuk_empty_grid(0, 256, 0, None) == 0
    assert L.gpuk_set_tuning(b"no_such_knob", 1) == 1 and L.gpuk_set_tuning(b"norm_quant_nchunk", 3) == 1
    assert L.gpuk_set_tuning(b"norm_quant_nchunk", 0) == 0
    assert L.gpuk_set_tuning(b"norm_quant_launches", 3) == 1 and L.gpuk_set_tuning(b"norm_quant_launches", 0) == 0


def test_torch_library_registers_reference_schemas():
    import gpuk_amd as gpuk

    def schema(name):
        return str(getattr(torch.ops.gpuk, name).default._schema)

    assert schema("allreduce_rms") == (
        "gpuk::allreduce_rms(SymInt fptr, Tensor allreduce_in, Tensor residual_in, Tensor rms_gamma, "
        "Tensor residual_out, Tensor norm_out, Tensor scale_out, float eps, SymInt quant_type) -> ()")
    assert schema("fused_rope_rms") == (
        "gpuk::fused_rope_rms(Tensor qkv, Tensor qw, Tensor kw, Tensor cos_sin, Tensor positions, SymInt num_tokens, "
        "SymInt num_heads_q, SymInt num_heads_k, SymInt num_heads_v, SymInt head_size, bool is_neox_style, "
        "float eps) -> ()")
    assert "int[] mrope_section_, bool is_interleaved, float eps) -> ()" in schema("fused_mrope_3d_rms")
    assert schema("fused_mrope_3d_rms_set_kv").endswith(
        "float eps, Tensor q, Tensor k_cache, Tensor v_cache, Tensor kv_loc, float k_scale, float v_scale) -> ()")
    for name in ("allreduce_rms", "fused_rope_rms", "fused_mrope_3d_rms", "fused_mrope_3d_rms_set_kv",
                 "fused_rope_rms_2way", "fused_rope_rms_set_kv", "set_fp8_max", "get_fp8_max"):
        assert hasattr(gpuk, name)
    assert gpuk.fp8 == torch.float8_e4m3fn and gpuk.fp8_max_val == 448 and gpuk.fp8_policy_id == 1


def test_two_way_op_has_a_meta_kernel():
    """Shape inference without a device, as the reference registers it (src/register.cpp:62-63)."""
    import gpuk_amd as gpuk

    m = lambda *s: torch.empty(*s, dtype=torch.bfloat16, device="meta")
    B, T0, T1, Hq, Hk, D = 2, 5, 7, 3, 2, 64
    q01, k01 = gpuk.fused_rope_rms_2way(m(B, T0, Hq, D), m(B, T0, Hk, D), m(B, T1, Hq, D), m(B, T1, Hk, D), m(D), m(D),
                                        m(D), m(D), m(T0, D), m(T1, D), B, T0, T1, Hq, Hk, D, False, 1e-6)
    assert q01.shape == (B, T0 + T1, Hq, D) and k01.shape == (B, T0 + T1, Hk, D)
    assert q01.device.type == "meta" and q01.dtype == torch.bfloat16
    assert str(torch.ops.gpuk.fused_rope_rms_2way.default._schema).endswith(
        "SymInt head_size, bool is_interleaved, float eps) -> (Tensor out_q01, Tensor out_k01)")


def test_fp8_max_setter_round_trip():
    import gpuk_amd as gpuk

    assert gpuk.get_fp8_max() == 448.0
    gpuk.set_fp8_max(240.0)
    try:
        assert gpuk.get_fp8_max() == 240.0
        with pytest.raises(RuntimeError):
            gpuk.set_fp8_max(0.0)
        with pytest.raises(RuntimeError):
            gpuk.set_fp8_max(1000.0)
    finally:
        gpuk.set_fp8_max(448.0)


def test_ops_refuse_cpu_tensors():
    """There is no CPU fallback: the compute ops exist for GPU tensors only."""
    import gpuk_amd as gpuk

    x = torch.zeros((2, 64), dtype=torch.bfloat16)
    with pytest.raises((RuntimeError, NotImplementedError)):
        gpuk.allreduce_rms(0, x, x, x[0], x.clone(), x.clone(), torch.zeros(2, 1), 1e-6, 0)
    with pytest.raises((RuntimeError, NotImplementedError)):
        gpuk.fused_rope_rms(torch.zeros((2, 3, 64), dtype=torch.bfloat16), x[0], x[0], torch.zeros((8, 64), dtype=torch.bfloat16),
                            torch.zeros(2, dtype=torch.int64), 2, 1, 1, 1, 64, True, 1e-6)


def test_algorithmic_byte_formulas():
    """Compulsory traffic per call, as published for the five configurations."""
    from gpuk_amd import workloads as W

    assert W.norm_quant_bytes(8192, 8192, 1) == 469_811_200
    assert W.norm_quant_bytes(128, 4096, 3) == 3_678_212
    assert [W.norm_quant_bytes(t, 7168, 1) for t in W.DECODE_TOKENS] == [64_516, 415_776, 1_620_096, 6_437_376, 25_706_496]
    assert W.rope_set_kv_bytes(4096, 32, 8, 8, 128, 1, 2) == 101_777_920
    assert W.rope_set_kv_bytes(8192, 28, 4, 4, 128, 3, 2) == 153_354_752
    assert W.rope_set_kv_bytes(1, 64, 8, 8, 128, 1, 1) == 39_696 and W.rope_set_kv_bytes(512, 64, 8, 8, 128, 1, 1) == 20_062_720
    # in-place form: the reference's own formula (test/cpp/test_rope_rms.cpp:184-188) plus the position read
    T, hq, hk, D = 513, 32, 32, 128
    ref = T * (hq + hk) * D * 2 + 2 * D * 2 + T * D * 2 + T * (hq + hk) * D * 2
    assert W.rope_inplace_bytes(T, hq, hk, D) == ref + 8 * T


def test_workload_generators_are_deterministic_and_shaped():
    from gpuk_amd import workloads as W

    a, b = W.config1(), W.config1()
    assert torch.equal(a.x, b.x) and a.x.shape == (128, 4096) and a.x.dtype == torch.bfloat16
    c2 = W.config2(64, 512)
    frac = (c2.x.abs() == 50).float().mean().item()
    assert 0.005 < frac < 0.015
    c3 = W.config3(256)
    assert c3.qkv.shape == (256, 48, 128) and c3.kv_loc.unique().numel() == 256 and c3.num_slots == 65536
    assert c3.cos_sin.shape == (32768, 128) and c3.cos_sin[0, :64].eq(1).all() and c3.cos_sin[0, 64:].eq(0).all()
    c4 = W.config4(4096)
    pos = c4.positions
    assert pos.shape == (3, 4096) and (pos[:, :1024] == torch.arange(1024)).all()
    img = pos[:, 1024:2048]
    assert (img[0] == 1024).all() and img[1].max() == 1024 + 31 and img[2].max() == 1024 + 31
    assert (pos[:, 2048] == 1024 + 32).all() and c4.mrope_section == [16, 24, 24]
    c5 = W.config5_rope(8)
    assert c5.kv_dtype == torch.float8_e4m3fn and c5.qkv.shape == (8, 80, 128)


def test_dist_env_rejects_multi_gpu_groups(monkeypatch):
    import torch.distributed as dist

    import gpuk_amd as gpuk

    monkeypatch.setattr(dist, "is_initialized", lambda: True)
    monkeypatch.setattr(dist, "get_rank", lambda group=None: 0)
    monkeypatch.setattr(dist, "get_world_size", lambda group=None: 2)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    with pytest.raises(NotImplementedError):
        gpuk.GPUKDistEnv(device_id=0)


def test_build_command_needs_nothing_built(tmp_path):
    """Where the libraries are missing, importing the package names a command that gets as far as the compiler."""
    import shutil
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    shutil.copytree(os.path.join(root, "gpuk_amd"), tmp_path / "gpuk_amd", ignore=shutil.ignore_patterns("lib", "build", "__pycache__"))
    run = lambda *args: subprocess.run([sys.executable, *args], cwd=tmp_path, capture_output=True, text=True, env={**os.environ, "HIPCC": "/bin/false"})
    missing = run("-c", "import gpuk_amd")
    command = re.search(r"not built; run `python (.*?)`", missing.stderr)
    assert missing.returncode != 0 and command
    started = run(*command[1].split())
    assert started.returncode != 0 and "command failed: /bin/false" in started.stderr


def test_bench_refuses_more_than_one_gpu():
    import subprocess
    import sys

    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert r.returncode != 0 and "single-GPU" in r.stderr


def test_mut_overloads_differ_from_reference_schemas_only_in_alias_annotations():
    """Every in-place operator has an overload `.mut` whose schema, with the `(x!)` annotations removed, is the
    reference's string (src/register.cpp:37-55), and which declares at least one written tensor."""
    import re

    import gpuk_amd  # noqa: F401  (loads the library)

    for name in ("allreduce_rms", "fused_rope_rms", "fused_mrope_3d_rms", "fused_mrope_3d_rms_set_kv",
                 "fused_rope_rms_set_kv"):
        packet = getattr(torch.ops.gpuk, name)
        assert packet.overloads() == ["default", "mut"], name
        plain, annotated = str(packet.default._schema), str(packet.mut._schema)
        assert "!)" in annotated and "!)" not in plain
        assert re.sub(r"\([a-z]!\)", "", annotated).replace(name + ".mut(", name + "(") == plain
    written = {a.name for a in torch.ops.gpuk.allreduce_rms.mut._schema.arguments if a.alias_info and a.alias_info.is_write}
    assert written == {"residual_out", "norm_out", "scale_out"}
    written = {a.name for a in torch.ops.gpuk.fused_mrope_3d_rms_set_kv.mut._schema.arguments
               if a.alias_info and a.alias_info.is_write}
    assert written == {"q", "k_cache", "v_cache"}
    written = {a.name for a in torch.ops.gpuk.fused_rope_rms.mut._schema.arguments if a.alias_info and a.alias_info.is_write}
    assert written == {"qkv"}


def test_mut_overloads_have_meta_kernels():
    """On meta tensors the `.mut` overloads run (and do nothing); the reference-schema overloads have no Meta
    kernel and refuse, as in the reference."""
    import gpuk_amd

    x = torch.empty((4, 64), dtype=torch.bfloat16, device="meta")
    g = torch.empty((64,), dtype=torch.bfloat16, device="meta")
    codes = torch.empty((4, 64), dtype=torch.float8_e4m3fn, device="meta")
    scale = torch.empty((4, 1), device="meta")
    assert gpuk_amd.traceable.allreduce_rms(0, x, x, g, x, codes, scale, 1e-6, 1) is None
    with pytest.raises(NotImplementedError):
        gpuk_amd.allreduce_rms(0, x, x, g, x, codes, scale, 1e-6, 1)
    qkv = torch.empty((4, 6, 64), dtype=torch.bfloat16, device="meta")
    pos = torch.empty((4,), dtype=torch.int64, device="meta")
    assert gpuk_amd.traceable.fused_rope_rms(qkv, g, g, x, pos, 4, 2, 2, 2, 64, True, 1e-6) is None


def test_reference_kernel_library_exports_its_entry_points():
    """oracle/_ref/libgpuk_ref.so (the reference's own kernels, compiled where a reference checkout exists) loads and
    exports the four entry points the GPU tests call.  Skipped where it was never built."""
    from oracle import ref_kernels

    if not ref_kernels.available():
        pytest.skip("oracle/_ref/libgpuk_ref.so not built")
    import torch  # noqa: F401  (its HIP runtime first, as for the product library)

    L = ref_kernels.lib()
    for name in ("gpuk_ref_rope_rms", "gpuk_ref_mrope_rms_set_kv", "gpuk_ref_rope_rms_2way", "gpuk_ref_epilogue_rows"):
        assert hasattr(L, name), name
    # argument refusal happens before any launch
    assert L.gpuk_ref_epilogue_rows(None, None, None, None, None, None, 0, 4096, 1e-6, 1, None) == -1
    assert L.gpuk_ref_rope_rms(None, None, None, None, None, 0, 1, 1, 4, 2, 2, 2, 96, 1, None, 0, 1e-6, None) == -1


def test_launch_shape_report():
    """gpuk_add_rmsnorm_quant_launch_shape computes on the host: lanes per row and 16-byte chunks per lane of the launch
    the norm-quant entry point would make (no GPU needed)."""
    from gpuk_amd import capi

    assert capi.add_rmsnorm_quant_launch_shape(8192, 8192) == (512, 2)
    assert capi.add_rmsnorm_quant_launch_shape(512, 7168) == (448, 2)
    # 1025-2048 rows of 7168: too many for one round at two chunks per lane, not at four (half the lanes per row)
    assert capi.add_rmsnorm_quant_launch_shape(1024, 7168) == (448, 2)
    assert capi.add_rmsnorm_quant_launch_shape(1025, 7168) == (256, 4)
    assert capi.add_rmsnorm_quant_launch_shape(2048, 8192) == (256, 4)
    assert capi.add_rmsnorm_quant_launch_shape(2049, 8192) == (512, 2)
    # from 1.1 rounds to two the call is two launches; the report is the first one's (1280 of 2600 rows, 1536 of 3000)
    assert capi.add_rmsnorm_quant_launch_shape(2252, 8192) == (512, 2)
    assert capi.add_rmsnorm_quant_launch_shape(2600, 8192) == (256, 4)
    assert capi.add_rmsnorm_quant_launch_shape(3000, 7168) == (256, 4)
    assert capi.add_rmsnorm_quant_launch_shape(4097, 7168) == (448, 2)
    # workgroups of five waves: a compute unit takes five of them, not six
    assert capi.add_rmsnorm_quant_launch_shape(1280, 5120) == (320, 2)
    assert capi.add_rmsnorm_quant_launch_shape(1281, 5120) == (192, 4)
    assert capi.add_rmsnorm_quant_launch_shape(1, 4096) == (256, 2)
    lanes, chunks = capi.add_rmsnorm_quant_launch_shape(4, 65600 * 2)    # rows that do not stay in registers
    assert chunks == 0 and lanes % 64 == 0
    # fp32 / fp64: chunks of 4 elements, kept in registers up to 4 x 1024 of them
    assert capi.add_rmsnorm_quant_launch_shape(128, 1024, torch.float32) == (128, 2)
    assert capi.add_rmsnorm_quant_launch_shape(128, 1024, torch.float64) == (256, 1)
    assert capi.add_rmsnorm_quant_launch_shape(128, 8192, torch.float64) == (1024, 2)
    assert capi.add_rmsnorm_quant_launch_shape(128, 12288, torch.float32) == (768, 4)
    assert capi.add_rmsnorm_quant_launch_shape(128, 16392, torch.float32) == (1024, 0)
    L = capi.lib()
    import ctypes as C
    a, b = C.c_int(0), C.c_int(0)
    assert L.gpuk_add_rmsnorm_quant_launch_shape(0, 1024, 0, C.byref(a), C.byref(b)) == 1
    assert L.gpuk_add_rmsnorm_quant_launch_shape(4, 1027, 0, C.byref(a), C.byref(b)) == 2
    assert L.gpuk_add_rmsnorm_quant_launch_shape(4, 1024, 0, None, C.byref(b)) == 1
    # the query refuses what the entry point refuses: rows that are no multiple of 8 elements (whatever the dtype),
    # and a dtype value that names no format
    assert L.gpuk_add_rmsnorm_quant_launch_shape(4, 16388, 2, C.byref(a), C.byref(b)) == 2
    assert L.gpuk_add_rmsnorm_quant_launch_shape(4, 1024, 7, C.byref(a), C.byref(b)) == 2


def test_launch_shape_report_by_mode():
    """The shape of a call without codes is its own: rows of two waves of two chunks take one chunk per lane up to 640 of them and
    from 833 to 1024, where quantised ones do up to 1280; fp32 batches of two launches are cut by the rows' own rule."""
    from gpuk_amd import capi

    shape, bf16, f16, f32 = capi.add_rmsnorm_quant_launch_shape, torch.bfloat16, torch.float16, torch.float32
    for dtype in (bf16, f16):
        for tokens, quantised, plain in ((640, 1, 1), (641, 1, 2), (832, 1, 2), (833, 1, 1), (1024, 1, 1), (1025, 1, 2), (1280, 1, 2), (1281, 2, 2)):
            lanes = lambda n: (128 * 2 // n, n)
            for quant, n in ((0, plain), (1, quantised), (3, quantised)):
                assert shape(tokens, 2048, dtype, quant) == lanes(n), (tokens, quant, dtype)
    # wide fp32 rows: two launches from 88 to 90 % of the pieces' layers without codes, from 92 to 96 % with them
    assert shape(1408, 5120, f32, 0) == (320, 4) and shape(1408, 5120, f32, 1) == (640, 2)
    assert shape(2306, 4096, f32, 0) == (256, 4) and shape(2306, 4096, f32, 1) == (512, 2)
    assert shape(64, 4096, torch.float64, 0) == shape(64, 4096, torch.float64, 1)
    L = capi.lib()
    a, b = ctypes.c_int(0), ctypes.c_int(0)
    refs = ctypes.byref(a), ctypes.byref(b)
    assert L.gpuk_add_rmsnorm_quant_launch_shape(700, 2048, 0, *refs) == 0 and (a.value, b.value) == shape(700, 2048)   # a quantised call's
    assert L.gpuk_add_rmsnorm_quant_launch_shape_of(700, 2048, 0, 2, *refs) == 2    # e4m3fnuz is refused
    assert L.gpuk_add_rmsnorm_quant_launch_shape_of(700, 2048, 7, 0, *refs) == 2
    assert L.gpuk_add_rmsnorm_quant_launch_shape_of(0, 2048, 0, 0, *refs) == 1


def test_store_gate_report():
    """gpuk_add_rmsnorm_quant_store_gate: a layer of rows, one per compute unit, that has just begun counts for most of a full one,
    but only behind a full one; up to 256 rows wait for their own share of the reads (no GPU needed)."""
    import ctypes as C
    from gpuk_amd import capi

    ticks = lambda rows, row_bytes: int(2 * rows * row_bytes / 70000.0)
    gate, f32 = capi.add_rmsnorm_quant_store_gate, torch.float32
    for tokens, hidden, rows in ((128, 16384, 1.05), (256, 16384, 1.05), (128, 32768, 1.08), (200, 32768, 1.08), (256, 32768, 1.08), (64, 65536, 1.08), (256, 65536, 1.08)):
        for quant in (0, 1, 3):
            assert gate(tokens, hidden, torch.bfloat16, quant) == ticks(rows * tokens, 2 * hidden), (tokens, hidden, quant)
    assert gate(200, 12288, f32, 0) == ticks(1.08 * 200, 4 * 12288)
    # behind a full layer: 0.93 of whole layers for 16-bit rows of four chunks per lane, else 0.86 with codes and 0.82 without
    assert gate(257, 8192) == ticks(0.86 * 512, 16384) and gate(257, 8192, quant=0) == ticks(0.82 * 512, 16384)
    assert gate(513, 16384) == ticks(0.93 * 768, 32768) and gate(257, 32768) == ticks(0.93 * 512, 65536)
    assert gate(340, 8192, f32) == ticks(0.86 * 512, 32768) and gate(318, 5120, f32, 0) == ticks(0.82 * 512, 20480)
    # ... unless the rows themselves are more than that
    assert gate(512, 8192) == ticks(1.05 * 512, 16384) and gate(500, 32768) == ticks(1.08 * 500, 65536)
    # no gate: less than a quarter of a round, more than one, small fp32 batches, fp64, swept rows
    for args in ((1, 8192), (127, 16384), (8192, 8192), (64, 4096, f32), (512, 4096, torch.float64), (300, 16392, f32), (4, 65600 * 2)):
        assert gate(*args) == 0, args
    out = C.c_int(0)
    assert capi.lib().gpuk_add_rmsnorm_quant_store_gate(0, 1024, 0, 1, C.byref(out)) == 1
    assert capi.lib().gpuk_add_rmsnorm_quant_store_gate(4, 1024, 0, 1, None) == 1
    assert capi.lib().gpuk_add_rmsnorm_quant_store_gate(4, 1028, 0, 1, C.byref(out)) == 2
    assert capi.lib().gpuk_add_rmsnorm_quant_store_gate(4, 1024, 0, 2, C.byref(out)) == 2
    assert capi.lib().gpuk_add_rmsnorm_quant_store_gate(4, 1024, 7, 1, C.byref(out)) == 2


def test_launch_shape_of_forced_chunks():
    """fp32 rows have forms of one, two and four chunks per lane: a forced eight is four there, eight for 16-bit rows."""
    from gpuk_amd import capi

    capi.set_tuning("norm_quant_nchunk", 8)
    try:
        assert capi.add_rmsnorm_quant_launch_shape(64, 16384, torch.float32) == (1024, 4)
        assert capi.add_rmsnorm_quant_launch_shape(64, 1024, torch.float32) == (64, 4)
        assert capi.add_rmsnorm_quant_launch_shape(64, 16384) == (256, 8)
    finally:
        capi.set_tuning("norm_quant_nchunk", 0)


def test_launch_shape_of_small_batches():
    """One chunk per lane where it leaves the busiest SIMD fewer chunks and the compute units have a row or two; four where
    each has one row of three or four full waves of them."""
    from gpuk_amd import capi

    bf16, f16, f32 = torch.bfloat16, torch.float16, torch.float32
    shape, gate = capi.add_rmsnorm_quant_launch_shape, capi.add_rmsnorm_quant_store_gate
    for hidden, dtype, changes in (
            (2048, bf16, ((1, 1), (1280, 1), (1281, 2))), (1544, f16, ((1, 1), (1280, 1), (1281, 2))), (1536, bf16, ((1, 1), (9, 1))),
            (1024, f32, ((1, 2), (192, 2))), (2056, bf16, ((1, 1), (1200, 1))),
            (5120, bf16, ((1, 1), (256, 1), (512, 1), (513, 2))), (5120, f16, ((1, 1), (192, 1), (193, 2), (256, 2), (257, 1), (512, 1), (513, 2))),
            (5640, bf16, ((192, 1), (193, 2), (256, 2), (257, 1), (512, 1), (513, 2))), (2560, f32, ((1, 1), (192, 1), (193, 2), (300, 2))),
            (6144, f16, ((1, 1), (128, 1), (129, 4), (256, 4), (257, 1), (512, 1), (513, 2))), (6152, bf16, ((1, 1), (200, 1))),
            (8192, bf16, ((1, 2), (128, 2), (129, 4), (256, 4), (257, 2))), (7168, bf16, ((200, 2),)), (7680, bf16, ((200, 1),)), (4096, f32, ((200, 2),))):
        chunks = hidden * (4 if dtype == f32 else 2) // 16
        for tokens, n in changes:
            lanes = (-(-chunks // n) + 63) // 64 * 64
            assert shape(tokens, hidden, dtype) == (lanes, n), (tokens, hidden, dtype)
    # one chunk per lane: stores wait from three eighths of a round, ten waves a row not in the first layer, one wave in half
    # precision without codes from a quarter
    for tokens, hidden, dtype, quant, waits in ((3071, 512, bf16, 1, False), (3072, 512, bf16, 1, True), (2048, 512, f16, 0, True), (2047, 512, f16, 0, False),
                                                (2048, 512, f16, 3, False), (256, 5120, bf16, 1, False), (257, 5120, bf16, 1, True),
                                                (191, 5632, bf16, 0, False), (192, 5632, bf16, 0, True), (512, 2048, bf16, 1, False), (1280, 2048, bf16, 1, True),
                                                (832, 2048, bf16, 0, False), (833, 2048, bf16, 0, True), (1024, 2048, bf16, 0, True)):
        assert (gate(tokens, hidden, dtype, quant) > 0) == waits, (tokens, hidden, dtype, quant)


def test_launch_shape_of_short_rows():
    """Rows that one wave holds with one chunk per lane keep that shape at every batch size."""
    from gpuk_amd import capi

    for tokens in (1, 8192, 8193, 9000, 100000):
        for hidden in (8, 128, 264, 512):
            assert capi.add_rmsnorm_quant_launch_shape(tokens, hidden) == (64, 1), (tokens, hidden)
        assert capi.add_rmsnorm_quant_launch_shape(tokens, 256, torch.float32) == (64, 1)
    assert capi.add_rmsnorm_quant_launch_shape(9000, 520) == (64, 2)


def test_launch_shape_of_thin_rows():
    """Rows of a little more than two waves' chunks, which two chunks per lane would leave a third of the lanes idle for:
    one chunk per lane from two waves' round to three of three waves, and in bfloat16 just above the latter's round."""
    from gpuk_amd import capi

    shape = capi.add_rmsnorm_quant_launch_shape
    assert [shape(t, 1032)[1] for t in (2560, 2561, 2880, 2881, 4096, 4097, 7680, 7681)] == [1, 1, 1, 2, 2, 1, 1, 2]
    assert [shape(t, 1032, torch.float16)[1] for t in (2560, 2561, 4096, 4097, 7680, 7681)] == [1, 2, 2, 1, 1, 2]
    assert [shape(t, 1360)[1] for t in (2560, 2561, 4097, 7680, 7681)] == [1, 2, 1, 1, 2]
    assert [shape(t, 516 + 4, torch.float32)[1] for t in (2560, 2561, 4097, 7681)] == [1, 2, 2, 2]
    assert [shape(t, 2056)[1] for t in (1280, 1281, 2561, 5000)] == [1, 2, 2, 2]


def test_launch_shape_of_two_launches():
    """Batches of one to two rounds run as two launches where the pieces idle at most a fifth of their lanes and the batch
    is more than a quarter over the round (the report is the first piece's: four chunks per lane instead of two)."""
    from gpuk_amd import capi

    assert capi.add_rmsnorm_quant_launch_shape(3200, 5120) == (320, 2)
    assert capi.add_rmsnorm_quant_launch_shape(3201, 5120) == (192, 4)
    assert capi.add_rmsnorm_quant_launch_shape(5120, 5120) == (192, 4)
    assert capi.add_rmsnorm_quant_launch_shape(5121, 5120) == (320, 2)
    assert capi.add_rmsnorm_quant_launch_shape(4608, 5120, torch.float16) == (192, 4)
    assert capi.add_rmsnorm_quant_launch_shape(11878, 1664) == (64, 4)
    assert capi.add_rmsnorm_quant_launch_shape(11878, 832, torch.float32) == (128, 2)   # fp32 rows of one wave: full ones only
    assert capi.add_rmsnorm_quant_launch_shape(12289, 1600) == (64, 4)                  # one wave: a quarter idle, from 1.5 rounds
    assert capi.add_rmsnorm_quant_launch_shape(5800, 3072) == (192, 2)                  # ... but not two waves
    # wide fp32 rows: one launch
    assert capi.add_rmsnorm_quant_launch_shape(1400, 7168, torch.float32) == (896, 2)
    assert capi.add_rmsnorm_quant_launch_shape(1600, 5120, torch.float32) == (640, 2)
    assert capi.add_rmsnorm_quant_launch_shape(2600, 3584, torch.float32) == (448, 2)
    # wide fp32 rows that fill the layers of workgroups of both launches
    assert capi.add_rmsnorm_quant_launch_shape(1518, 5120, torch.float32) == (320, 4)
    assert capi.add_rmsnorm_quant_launch_shape(1531, 8192, torch.float32) == (512, 4)
    assert capi.add_rmsnorm_quant_launch_shape(2020, 7168, torch.float32) == (448, 4)
    assert capi.add_rmsnorm_quant_launch_shape(2700, 4096, torch.float32) == (256, 4)


def test_rope_launch_shape_report():
    """gpuk_rope_rms_launch_shape computes on the host which rope kernel a batch gets, its grid and whether the rotated
    rows are stored past the L2; no GPU is needed."""
    from gpuk_amd import capi
    # 4096 tokens x (32, 8, 8) heads of 128 with a 16-bit cache: the batch fits the chip in one round, one wave per token
    assert capi.rope_rms_launch_shape(4096, 32, 8, 8, 128) == (1024, 256, True, 1)
    # 4200 tokens do not: one wave per group of 8 Q/K heads, four waves a workgroup, streamed stores
    assert capi.rope_rms_launch_shape(4200, 32, 8, 8, 128) == (5250, 256, True, False)
    assert capi.rope_rms_launch_shape(4096, 32, 8, 8, 128, set_kv=False) == (1024, 256, True, 1)   # in place too
    assert capi.rope_rms_launch_shape(2048, 32, 8, 8, 128, set_kv=False) == (2560, 256, True, 0)
    # 8192 tokens of 28+4+4 heads: two tokens per wave, the second through LDS, still one round
    assert capi.rope_rms_launch_shape(8192, 28, 4, 4, 128, n_axes=3) == (1024, 256, True, 2)
    assert capi.rope_rms_launch_shape(8192, 28, 4, 4, 128, n_axes=3, set_kv=False) == (1024, 256, True, 2)
    assert capi.rope_rms_launch_shape(4096, 32, 8, 8, 128, kv_fp8=True) == (1024, 256, True, 1)
    assert capi.rope_rms_launch_shape(2560, 32, 8, 8, 128, kv_fp8=True) == (3200, 256, True, 0)   # an fp8 cache: later
    # a decode batch: through the L2; single waves unless a workgroup of four holds whole tokens
    assert capi.rope_rms_launch_shape(16, 28, 4, 4, 128) == (16, 256, False, False)
    assert capi.rope_rms_launch_shape(16, 40, 8, 8, 128, kv_fp8=True) == (96, 64, False, False)
    # fp32 activations: a wave per 512/D Q/K heads, and per 512 elements of the V row when a cache is written
    assert capi.rope_rms_launch_shape(10, 4, 2, 2, 64, dtype=torch.float32) == (5, 256, True, False)
    assert capi.rope_rms_launch_shape(10, 4, 2, 2, 64, dtype=torch.float32, set_kv=False) == (3, 256, True, False)
    assert capi.rope_rms_launch_shape(4, 7, 2, 3, 256, dtype=torch.float64) == (7, 256, True, False)
    import ctypes as C
    L = capi.lib()
    o = [C.c_int(0) for _ in range(4)]
    refs = [C.byref(x) for x in o]
    assert L.gpuk_rope_rms_launch_shape(0, 32, 8, 8, 128, 1, 0, 1, 0, *refs) == 1
    assert L.gpuk_rope_rms_launch_shape(4, 32, 8, 8, 96, 1, 0, 1, 0, *refs) == 2
    assert L.gpuk_rope_rms_launch_shape(4, 32, 8, 8, 128, 2, 0, 1, 0, *refs) == 1
    assert L.gpuk_rope_rms_launch_shape(4, 32, 8, 8, 128, 1, 0, 1, 0, None, *refs[1:]) == 1
    assert L.gpuk_rope_rms_launch_shape(4, 32, 8, 8, 128, 1, 9, 1, 0, *refs) == 2   # no such dtype


def test_rope_launch_shape_report_of_rotation_and_sections():
    """The report answers for the rotation and the sections it is given: the kernel's choice depends on both."""
    from gpuk_amd import capi

    shape = lambda T, **kw: capi.rope_rms_launch_shape(T, 28, 4, 4, 128, 3, **kw)
    assert shape(4608) == shape(4608, mrope_section=[16, 24, 24]) and shape(4608)[3] == 2
    assert shape(2400, is_neox=False) == shape(2400) and shape(2400)[3] == 0              # whole tokens of four: from five quarters of a round
    assert shape(2400, mrope_section=[24, 20, 20], is_interleaved=True)[3] == 1           # three table rows: from nine eighths
    assert shape(3100)[3] == 1 and shape(3100, is_neox=False)[3] == 0                     # a layer of waves that has just begun
    assert shape(4200)[3] == 0                                                            # two whole tokens of four: from 4608
    assert shape(4200, is_neox=False, mrope_section=[24, 20, 20], is_interleaved=True)[3] == 2   # three table rows pairwise: at once
    assert capi.rope_rms_launch_shape(1850, 64, 64, 64, 64, is_neox=False)[1] == 256
    # in place, parts of a token: a form for rotation by halves only
    assert capi.rope_rms_launch_shape(1536, 40, 8, 8, 128, set_kv=False)[3] == 1
    assert capi.rope_rms_launch_shape(1536, 40, 8, 8, 128, set_kv=False, is_neox=False)[3] == 0
    L = capi.lib()
    outs = [ctypes.c_int(0) for _ in range(4)]
    refs = [ctypes.byref(o) for o in outs]
    bad = (ctypes.c_int64 * 3)(16, 24, 23)
    assert L.gpuk_rope_rms_launch_shape_of(64, 28, 4, 4, 128, 3, 0, 1, 0, 1, bad, 0, *refs) == 1   # sections that do not fill a head
    assert L.gpuk_rope_rms_launch_shape_of(64, 28, 4, 4, 128, 1, 0, 1, 0, 1, bad, 0, *refs) == 0   # (one axis: not looked at)
    for T in (64, 1400, 4096, 8192):
        assert L.gpuk_rope_rms_launch_shape(T, 28, 4, 4, 128, 3, 0, 1, 0, *refs) == 0
        assert (outs[0].value, outs[1].value, bool(outs[2].value), outs[3].value) == shape(T)


def test_rope_kernel_choice():
    """Which calls the kernel with one wave per token or part of one takes (1: one item per wave, 2: two), from both sides of
    the lines of its rule: rotation by halves, then pairwise."""
    from gpuk_amd import capi

    bf16, f16 = torch.bfloat16, torch.float16
    for heads, D, dtype, cache, halves, pairwise in (
            # (tokens, which kernel from there on, at every change up to 8400)
            # three units per item: beyond a round of the other kernel's waves; half precision from seven eighths, by halves where lanes are full
            ((16, 2, 2), 128, bf16, True, ((2731, 1), (3073, 0), (3328, 1), (4097, 0), (4608, 2), (5121, 0), (5632, 2), (6145, 0), (6656, 2), (7169, 0), (7680, 2), (8193, 0)),
             ((2731, 1), (3073, 0), (3328, 1), (4097, 0), (4608, 2), (5121, 0), (5632, 2), (6145, 0), (6656, 2), (7169, 0))),
            ((16, 2, 2), 128, f16, True, ((2731, 1), (3073, 0), (3328, 1), (4097, 2), (8193, 0)), ((2390, 1), (3073, 0), (3712, 1), (4097, 2), (7169, 0))),
            ((12, 12, 12), 128, bf16, True, ((2731, 1), (4097, 0)), ((2731, 1), (3073, 0), (3712, 1), (4097, 0))),
            ((12, 12, 12), 128, f16, True, ((2390, 1), (4097, 0)), ((2390, 1), (3073, 0), (3328, 1), (4097, 0))),
            ((24, 8, 8), 256, bf16, True, ((1152, 1), (2049, 0)), ((1152, 1), (1537, 0), (1664, 1), (2049, 0))),
            # four, five: bfloat16 from nine eighths of a round, whole tokens of four and five with idle units from five quarters
            ((28, 4, 4), 256, bf16, True, ((1152, 1), (2049, 2), (4097, 0)), ((1152, 1), (1537, 0), (1664, 1), (2049, 2), (3585, 0))),
            ((28, 4, 4), 128, bf16, True, ((2560, 1), (4097, 0), (4608, 2), (8193, 0)), ((2560, 1), (3073, 0), (3328, 1), (4097, 0), (4608, 2), (7169, 0))),
            ((28, 4, 4), 128, f16, True, ((1792, 1), (4097, 2), (8193, 0)), ((1792, 1), (3073, 0), (3328, 1), (4097, 2), (7169, 0))),
            ((32, 8, 8), 128, bf16, True, ((1844, 1), (4097, 0)), ((1844, 1), (3073, 0), (3328, 1), (4097, 0))),
            ((32, 8, 8), 128, f16, True, ((1536, 1), (4097, 0)), ((1536, 1), (3073, 0), (3328, 1), (4097, 0))),
            ((96, 12, 12), 128, bf16, True, ((732, 1), (1366, 2), (2049, 0)), ((732, 1), (1025, 0), (1110, 1), (1366, 2), (1434, 0), (1639, 2), (1793, 0))),
            # in place; pairwise whole tokens only
            ((32, 8, 8), 128, bf16, False, ((2458, 1), (3073, 0), (3328, 1), (4097, 0)), ((2458, 1), (3073, 0), (3328, 1), (4097, 0))),
            ((28, 4, 4), 128, bf16, False, ((2816, 1), (3073, 0), (3328, 1), (4097, 0), (4608, 2), (8193, 0)), ((2816, 1), (3073, 0), (3328, 1), (4097, 0), (4608, 2), (7169, 0))),
            ((28, 4, 4), 128, f16, False, ((1920, 1), (4097, 2), (8193, 0)), ((1792, 1), (3073, 0), (3712, 1), (4097, 2), (7169, 0))),
            ((16, 2, 2), 128, f16, False, ((2731, 1), (3073, 0), (3328, 1), (4097, 2), (7169, 0)), ()),
            ((12, 12, 12), 128, f16, False, ((2390, 1), (4097, 2), (7169, 0)), ())):
        for changes, neox in ((halves, True), (pairwise, False)):
            kernel = lambda T: capi.rope_rms_launch_shape(T, *heads, D, 1, dtype, cache, False, neox)[3]
            was = 0
            for tokens, expect in changes:
                assert (kernel(tokens - 1), kernel(tokens)) == (was, expect), (tokens, heads, D, dtype, cache, neox)
                was = expect
            last = changes[-1][0] if changes else 300
            assert all(kernel(T) == was for T in range(last, 8400, 101)), (heads, D, dtype, cache, neox)
    # an fp8 cache: whole tokens, not where the last layer of waves has just begun
    for tokens, heads, expect in ((2560, (28, 4, 4), 1), (3200, (28, 4, 4), 0), (3328, (28, 4, 4), 1), (2662, (32, 8, 8), 0), (2663, (32, 8, 8), 1), (3100, (32, 8, 8), 0)):
        assert capi.rope_rms_launch_shape(tokens, *heads, 128, 1, bf16, True, True)[3] == expect, (tokens, heads)


def test_rope_workgroups():
    """Lanes per workgroup of the rope kernel with one wave per group of heads: four waves in place in bfloat16 by halves from five eighths of
    a round of waves and behind the gate of heads of 64 that fill their lanes, in other forms from two thirds, in whole lines behind a gate, and single waves
    where an fp8 cache of many V heads keeps the vector units busy and for tokens of three units just beyond a round."""
    from gpuk_amd import capi

    bf16, f16 = torch.bfloat16, torch.float16
    for tokens, heads, dtype, neox, lanes in ((1023, (32, 8, 8), bf16, True, 64), (1024, (32, 8, 8), bf16, True, 256), (1092, (32, 8, 8), bf16, False, 64), (1093, (32, 8, 8), bf16, False, 256),
                                              (1092, (32, 8, 8), f16, True, 64), (1093, (32, 8, 8), f16, True, 256), (1820, (16, 2, 2), f16, False, 64), (1821, (16, 2, 2), f16, False, 256)):
        assert capi.rope_rms_launch_shape(tokens, *heads, 128, 1, dtype, False, False, neox)[1] == lanes, (tokens, heads, dtype, neox)
    for T, neox, lanes in ((1535, True, 64), (1536, True, 256), (2047, False, 64), (2048, False, 256)):   # two fifths of the lanes idle
        assert capi.rope_rms_launch_shape(T, 8, 1, 1, 128, 1, bf16, False, False, neox)[1] == lanes, (T, neox)
    for heads, changes in (((72, 8, 8), 820), ((64, 8, 8), 1093)):   # (lanes that idle: from two thirds)
        assert [capi.rope_rms_launch_shape(T, *heads, 64, 1, bf16, False, False, False)[1] for T in (changes - 1, changes)] == [64, 256]
    for tokens, heads, D, dtype, cache, fp8, lanes in (
            (1023, (64, 8, 8), 64, bf16, False, False, 64), (1024, (64, 8, 8), 64, bf16, False, False, 256), (1092, (64, 8, 8), 64, f16, False, False, 64),
            (1706, (32, 8, 8), 64, bf16, True, False, 64), (1707, (32, 8, 8), 64, bf16, True, False, 256), (1707, (32, 8, 8), 64, f16, True, False, 64),
            (255, (64, 64, 64), 128, bf16, True, True, 256), (256, (64, 64, 64), 128, bf16, True, True, 64), (512, (64, 64, 64), 128, bf16, True, True, 64),
            (513, (64, 64, 64), 128, bf16, True, True, 256), (2000, (16, 16, 16), 128, bf16, True, True, 256),
            (2730, (40, 8, 8), 64, bf16, True, False, 256), (2731, (40, 8, 8), 64, bf16, True, False, 64), (4096, (16, 2, 2), 128, bf16, True, True, 64),
            (4097, (16, 2, 2), 128, bf16, True, True, 256), (2731, (40, 8, 8), 64, bf16, False, False, 256)):
        assert capi.rope_rms_launch_shape(tokens, *heads, D, 1, dtype, cache, fp8)[1] == lanes, (tokens, heads, D, dtype, cache, fp8)
