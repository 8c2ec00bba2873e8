"""The operators' names in the package call past the interpretation of the schema where the arguments are plain: what they
return, raise and let others see is what the general call of the same packet gives (no GPU needed: meta tensors)."""
import inspect
import types

import pytest
import torch
from torch._subclasses import FakeTensorMode
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
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    for mode in (Functions, Dispatch):
        for f in (packet, general(packet)):
            seen.clear()
            with mode():
                f(*args)
            assert [str(s) for s in seen if "gpuk" in str(s)] == ["gpuk.fused_rope_rms_2way.default"] or mode is Functions, (mode, seen)
            assert any("fused_rope_rms_2way" in str(s) for s in seen), (mode, seen)
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
