"""The operators' names in the package call past the interpretation of the schema where the arguments are plain: what they
return, raise and let others see is what the general call of the same packet gives (no GPU needed: meta tensors)."""
import inspect
import types

import pytest
import torch
from torch._subclasses import FakeTensorMode
from torch.autograd import forward_ad
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

import gpuk_amd as gpuk

B, T0, T1, H, D = 2, 3, 5, 4, 64
NAMES = ["allreduce_rms", "fused_rope_rms", "fused_mrope_3d_rms", "fused_mrope_3d_rms_set_kv", "fused_rope_rms_set_kv", "fused_rope_rms_2way"]


def general(packet):
    return types.MethodType(torch._ops.OpOverloadPacket.__call__, packet)


def two_way(device="meta", dtype=torch.bfloat16, **kw):
    new = lambda *shape: torch.zeros(shape, dtype=dtype, device=device, **kw)
    return (new(B, T0, H, D), new(B, T0, H, D), new(B, T1, H, D), new(B, T1, H, D), *[new(D) for _ in range(4)], new(T0, D), new(T1, D),
            B, T0, T1, H, H, D, True, 1e-6)


def outcome(f, *args, **kw):
    try:
        out = f(*args, **kw)
    except Exception as e:   # noqa: BLE001  (the point is that both raise the same)
        return type(e), str(e)
    return type(out), [(t.shape, t.dtype, t.device, t.requires_grad, type(t)) for t in out] if out is not None else None


@pytest.mark.parametrize("name", NAMES)
def test_the_packet_stays_what_it_was(name):
    packet = getattr(gpuk, name)
    assert packet is getattr(torch.ops.gpuk, name)
    assert isinstance(packet, torch._ops.OpOverloadPacket) and str(packet) == f"gpuk.{name}"
    assert packet.default._schema.name == f"gpuk::{name}"
    assert inspect.signature(packet) == inspect.signature(general(packet))


@pytest.mark.parametrize("name", NAMES)
def test_wrapped_once_more(name):
    """As where the module is executed again: keyword calls must still reach the packet's own call, with its own arguments."""
    packet = getattr(gpuk, name)
    expect = outcome(general(packet), **{"eps": 1e-6})
    assert gpuk._called_directly(packet) is packet
    assert outcome(packet, **{"eps": 1e-6}) == expect
    if name == "fused_rope_rms_2way":
        args = two_way()
        assert outcome(packet, *args[:17], eps=1e-6) == outcome(packet, *args) == outcome(general(packet), *args)


def arguments(name, device="meta", dtype=torch.bfloat16):
    """Plain arguments of every function that calls an operator directly."""
    new = lambda *shape, dt=dtype: torch.zeros(shape, dtype=dt, device=device)
    tokens, hq, hk, hv = 5, 4, 2, 2
    if name == "allreduce_rms":
        return 0, new(tokens, 64), new(tokens, 64), new(64), new(tokens, 64), new(tokens, 64), new(tokens, 1, dt=torch.float32), 1e-6, 0
    if name == "add_rms_fused":
        return new(tokens, 64), new(tokens, 64), new(64), 1e-6, 1
    if name == "add_rms_fused.static":
        return new(tokens, 64), new(tokens, 64), new(64), 1e-6, new(1, dt=torch.float32)
    if name == "fused_rope_rms_2way":
        return two_way(device, dtype)
    axes = (3,) if "mrope" in name else ()
    args = (new(tokens, hq + hk + hv, D), new(D), new(D), new(16, D), new(*axes, tokens, dt=torch.int64), tokens, hq, hk, hv, D, True)
    args += ([8, 12, 12], False, 1e-6) if axes else (1e-6,)
    if "set_kv" in name:
        args += (new(tokens, hq, D), new(32, hk, D), new(32, hv, D), new(tokens, dt=torch.int64), 0.5, 0.25)
    return args


def both(name):
    """(direct function, general one) of an entry of the table in csrc/direct_calls.cpp."""
    if name == "add_rms_fused":
        return gpuk._add_rms_fused_direct, gpuk._add_rms_fused
    if name == "add_rms_fused.static":
        return gpuk._add_rms_fused_static_direct, gpuk._add_rms_fused_static
    return getattr(gpuk, name), general(getattr(gpuk, name))


ENTRIES = NAMES + ["add_rms_fused", "add_rms_fused.static"]


class recorded:
    """Kernels of the CPU key for the length of a test, which note what reached the operator."""

    def __enter__(self):
        self.lib, self.calls = torch.library.Library("gpuk", "IMPL"), []
        for name in ENTRIES:
            def kernel(*args, name=name):
                self.calls.append((name, [(a.shape, a.dtype, a.data_ptr()) if torch.is_tensor(a) else (type(a), a) for a in args]))
                if "add_rms_fused" in name:
                    out = torch.ones_like(args[1]), torch.full_like(args[0], 2)
                    return out if "static" in name else (*out, torch.full((1,), 3.0))
                return (args[0] + 1, args[1] + 2) if "2way" in name else None
            self.lib.impl(name, kernel, "CPU")
        return self.calls

    def __exit__(self, *_):
        self.lib._destroy()


@pytest.mark.parametrize("name", ENTRIES)
def test_every_function_hands_on_its_arguments(name):
    direct, packet = both(name)
    args = arguments(name, "cpu")
    values = [7 + i if type(a) is int else 0.25 + i if type(a) is float else a for i, a in enumerate(args)]   # (each to be told apart)
    with recorded() as calls:
        out, expect = direct(*values), packet(*values)
        assert len(calls) == 2 and calls[0] == calls[1] and calls[0][0] == name
        assert [type(a) for a in values] == [a[0] if isinstance(a[0], type) else torch.Tensor for a in calls[0][1]]
    if expect is None:
        assert out is None
    else:
        assert type(out) is type(expect) and len(out) == len(expect) and all(torch.equal(a, b) for a, b in zip(out, expect))


@pytest.mark.parametrize("name", ENTRIES)
def test_every_function_raises_what_the_general_call_raises(name):
    direct, packet = both(name)
    meta, cpu = arguments(name), arguments(name, "cpu")
    assert outcome(direct, *meta) == outcome(packet, *meta)
    with recorded() as calls:
        for at, a in enumerate(cpu):
            for other in (None, "x", 1.5, 3, True, 2 ** 70, torch.tensor(2), [1, 2, 3], (1, 2, 3), [1, 2.0, 3], [1, True, 3], [1, 2 ** 70, 3], []):
                if name.endswith("static") and at == 4 and torch.is_tensor(other):
                    other = other.float()
                args = (*cpu[:at], other, *cpu[at + 1:])
                assert outcome(direct, *args) == outcome(packet, *args), (at, other)
        for args in (cpu[:-1], (*cpu, 1), ()):
            got, expect = outcome(direct, *args), outcome(packet, *args)
            assert got[0] == expect[0] and (got == expect or "static" in name), args   # (the message names a Python function there)
        # what arrived, arrived the same either way
        assert len(calls) % 2 == 0 and all(a == b for a, b in zip(calls[::2], calls[1::2]))


@pytest.mark.parametrize("sections", [[8, 12, 12], (8, 12, 12), torch.Size([8, 12, 12]), [], [1, 2], [2 ** 62, -1, 0]])
@pytest.mark.parametrize("name", ["fused_mrope_3d_rms", "fused_mrope_3d_rms_set_kv"])
def test_sections(name, sections):
    direct, packet = both(name)
    args = [sections if type(a) is list else a for a in arguments(name, "cpu")]
    with recorded() as calls:
        direct(*args), packet(*args)
        assert calls[0] == calls[1] and (list, list(sections)) in calls[0][1]


@pytest.mark.parametrize("shape", [(), (1,), (1, 1)])
def test_the_static_scale_is_the_third_output(shape):
    args = (*arguments("add_rms_fused.static", "cpu")[:4], torch.full(shape, 0.5))
    with recorded():
        for f in both("add_rms_fused.static"):
            out = f(*args)
            assert len(out) == 3 and out[2].shape == (1,) and out[2].data_ptr() == args[4].data_ptr()


@pytest.mark.parametrize("change", [
    {}, {10: 1.5}, {10: True}, {16: 1}, {17: 0}, {0: None}, {11: 2 ** 70}, {"cut": 17}, {"add": 3}, {"device": "cpu"},
    {"requires_grad": True}, {0: torch.nn.Parameter(torch.zeros(B, T0, H, D, device="meta"))}])
def test_plain_and_other_arguments(change):
    packet = gpuk.fused_rope_rms_2way
    args = list(two_way(change.get("device", "meta"), **({"requires_grad": True} if "requires_grad" in change else {})))
    for at, value in change.items():
        if isinstance(at, int):
            args[at] = value
    args = args[:change.get("cut", len(args))] + ([change["add"]] if "add" in change else [])
    assert outcome(packet, *args) == outcome(general(packet), *args)


def test_keywords_and_subclasses():
    packet, args = gpuk.fused_rope_rms_2way, two_way()
    names = [a.name for a in packet.default._schema.arguments]
    assert outcome(packet, **dict(zip(names, args))) == outcome(packet, *args)
    assert outcome(packet, *args[:17], eps=1e-6) == outcome(packet, *args)

    class Marked(torch.Tensor):
        seen = 0

        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            Marked.seen += 1
            return super().__torch_function__(func, types, args, kwargs or {})

    marked = (args[0].as_subclass(Marked), *args[1:])
    assert outcome(packet, *marked) == outcome(general(packet), *marked) and Marked.seen >= 2


def test_modes_see_the_call():
    packet, args = gpuk.fused_rope_rms_2way, two_way()
    seen = []

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    for mode in (Functions, Dispatch):
        records = []
        for f in (packet, general(packet)):
            seen.clear()
            with mode():
                f(*args)
            records.append(list(seen))
        assert records[0] == records[1] and any("fused_rope_rms_2way" in s for s in records[0]), (mode, records)
    assert records[0][0] == "gpuk.fused_rope_rms_2way.default"
    with FakeTensorMode():
        out = packet(*two_way("cuda"))
    assert out[0].device.type == "cuda" and out[0].shape == (B, T0 + T1, H, D)


def test_vmap_compile_and_profiler():
    packet, args = gpuk.fused_rope_rms_2way, two_way()
    batched = lambda f: torch.vmap(lambda q0: f(q0, *args[1:]))(torch.zeros(2, B, T0, H, D, dtype=torch.bfloat16, device="meta"))
    assert outcome(batched, packet) == outcome(batched, general(packet))
    nodes = []

    def backend(graph, inputs):
        nodes.extend(str(n.target) for n in graph.graph.nodes if n.op == "call_function")
        return graph.forward

    torch._dynamo.reset()
    out = torch.compile(lambda *a: packet(*a), backend=backend, fullgraph=True)(*args)
    assert out[0].shape == (B, T0 + T1, H, D) and any("fused_rope_rms_2way" in n for n in nodes), nodes
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        packet(*args)
    assert any(e.key == "gpuk::fused_rope_rms_2way" for e in prof.key_averages())
    scripted = torch.jit.trace(lambda q0: packet(q0, *args[1:])[0], args[0], check_trace=False)
    assert "gpuk::fused_rope_rms_2way" in str(scripted.graph)


@pytest.mark.gpu
@pytest.mark.parametrize("around", ["plain", "parameter", "parameter, no_grad", "inference", "dispatch mode", "functions mode", "vmap", "grad", "profiler", "fake", "dual", "jvp", "hooks", "autocast"])
def test_two_streams_on_the_gpu_around_autograd(device, around):
    """The operator returns tensors and has no derivative: outputs, their place in a graph, their tangents and what a mode, a
    profiler or saved-tensor hooks see are the general call's."""
    packet = gpuk.fused_rope_rms_2way
    gen = torch.Generator().manual_seed(3)
    args = tuple(torch.randn(a.shape, generator=gen).bfloat16().to(device) if torch.is_tensor(a) else a for a in two_way("cpu"))
    if "parameter" in around:
        args = (*args[:4], args[4].requires_grad_(), *args[5:])
    seen = []

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    def call(f):
        seen.clear()
        if around == "parameter, no_grad":
            with torch.no_grad():
                return f(*args)
        if around == "inference":
            with torch.inference_mode():
                return f(*args)
        if "mode" in around:
            with Dispatch() if "dispatch" in around else Functions():
                return f(*args)
        if around == "vmap":
            return torch.vmap(lambda q0: f(q0, *args[1:]))(torch.stack([args[0], args[0]]))
        if around == "grad":
            return torch.func.grad_and_value(lambda w: f(*args[:4], w, *args[5:])[0].float().sum())(args[4].float().bfloat16())
        if around == "dual":
            with forward_ad.dual_level():
                out = f(forward_ad.make_dual(args[0], torch.ones_like(args[0])), *args[1:])
                assert all(forward_ad.unpack_dual(t).tangent is None for t in out)
                return out
        if around == "jvp":
            return torch.func.jvp(lambda q0: f(q0, *args[1:]), (args[0],), (torch.ones_like(args[0]),))[0]
        if around == "hooks":
            with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append("saved") or t, lambda t: t):
                return f(*args[:4], args[4].clone().requires_grad_(), *args[5:])
        if around == "autocast":
            with torch.autocast("cuda", dtype=torch.float16):
                return f(*args)
        if around == "profiler":
            with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
                out = f(*args)
            assert any(e.key == "gpuk::fused_rope_rms_2way" for e in prof.key_averages())
            return out
        if around == "fake":
            with FakeTensorMode(allow_non_fake_inputs=True) as mode:
                return f(*[mode.from_tensor(a) if torch.is_tensor(a) else a for a in args])
        return f(*args)

    def result(f):
        try:
            out = call(f)
        except Exception as e:   # noqa: BLE001
            return type(e), str(e)[:200], list(seen)
        flat = [t for t in out if torch.is_tensor(t)]
        return [(t.shape, t.dtype, str(t.device), t.requires_grad, type(t.grad_fn).__name__, t.is_inference(), type(t)) for t in flat], list(seen), flat

    got, want = result(packet), result(general(packet))
    assert got[:2] == want[:2], (got[:2], want[:2])
    if around != "fake" and isinstance(got[2], list) and got[2] and torch.is_tensor(got[2][0]):
        assert all(torch.equal(a, b) for a, b in zip(got[2], want[2]))


@pytest.mark.parametrize("name", [n for n in NAMES if "2way" not in n])
def test_in_place_operators_with_parameters(name):
    """They return nothing a graph could hold: weights that are parameters or duals change nothing, with gradients asked for or not."""
    direct, packet = both(name)
    args = [a.requires_grad_() if torch.is_tensor(a) and a.dim() == 1 and a.is_floating_point() else a for a in arguments(name, "cpu")]
    with recorded() as calls:
        for f in (direct, packet):
            assert f(*args) is None
            with torch.no_grad():
                assert f(*args) is None
        with forward_ad.dual_level():
            duals = [forward_ad.make_dual(a.detach(), torch.ones_like(a)) if torch.is_tensor(a) and a.requires_grad else a for a in args]
            for f in (direct, packet):
                assert f(*duals) is None
    assert len(calls) == 6 and all(c == calls[0] for c in calls[:4]) and calls[4] == calls[5]
    assert all(not torch.is_tensor(a) or a.grad_fn is None for a in args)


@pytest.mark.gpu
def test_capture_status(device):
    ask, torchs = gpuk._direct.current_stream_is_capturing, torch.cuda.is_current_stream_capturing
    assert ask() is torchs() is False
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert ask() is torchs() is False
    buf = torch.zeros(8, device=device)
    torch.cuda.synchronize()
    with torch.cuda.graph(torch.cuda.CUDAGraph()):
        assert ask() is torchs() is True
        buf.add_(1)
    assert ask() is torchs() is False


@pytest.mark.gpu
def test_capture_status_beside_a_captured_blocking_stream(device):
    """While a stream that blocks the null stream is captured, the runtime refuses to say that the null stream is not: the query and
    the env's call, which synchronises the device after a capture, pass that on as torch's query does."""
    import ctypes

    hip = ctypes.CDLL("libamdhip64.so")
    env = gpuk.GPUKDistEnv(device_id=torch.cuda.current_device())
    x = torch.randn(4, 1024, device=device).bfloat16()
    args = (x, x.clone(), torch.ones(1024, device=device, dtype=x.dtype), 1e-6)
    want = env.allreduce_add_rms_fused(*args, fp8_out=True)
    torch.cuda.synchronize()
    stream, graph = ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(stream), 0) == 0
    try:
        assert hip.hipStreamBeginCapture(stream, 1) == 0      # thread-local mode
        try:
            for ask in (torch.cuda.is_current_stream_capturing, gpuk._direct.current_stream_is_capturing, lambda: env.allreduce_add_rms_fused(*args, fp8_out=True)):
                with pytest.raises(RuntimeError, match="legacy stream"):
                    ask()
        finally:
            assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
            if graph:
                hip.hipGraphDestroy(graph)
    finally:
        torch.cuda.synchronize()
        assert hip.hipStreamDestroy(stream) == 0
    for a, b in zip(env.allreduce_add_rms_fused(*args, fp8_out=True), want):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
