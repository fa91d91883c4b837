"""The measuring entry points change nothing but the clock: a forward whose launches carry their own events
(rbmoe_forward_kernel_times), a forward with events between the stages (rbmoe_forward_timed) and the replay of one
stage (rbmoe_replay_stage) leave the same output bits and the same routing tables as a plain forward."""
import numpy as np
import pytest

from bench import DeviceBuffer
from conftest import rel_l2
from helpers import gpu_layer, last_products, small_workload
from rustingbrain_amd import _lib as L
from rustingbrain_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [dict(d=128, E=8, k=2, F=192, T=700, shared=True),     # large-batch kernels
                                   dict(d=128, E=8, k=2, F=192, T=16, shared=True),      # decode-shaped, routing beside
                                   dict(d=256, E=40, k=2, F=1152, T=8),                  # decode-shaped, routing in front
                                   dict(d=64, E=40, k=2, F=64, T=8)],                    # few slots, little to fetch for nothing
                         ids=["batch", "decode_front", "decode", "decode_front_few_slots"])
def test_measuring_entry_points_leave_the_results_alone(device, shape):
    t = synth.make(small_workload(seed=91, act="bf16", wt="bf16", **shape))
    T = shape["T"]
    layer = gpu_layer(device, t)
    x = synth.f32_to_bf16_bits(t.x)
    xb, ob = DeviceBuffer(device, x.nbytes).upload(x), DeviceBuffer(device, x.nbytes)

    def snapshot():
        device.synchronize()
        out = ob.download(np.empty_like(x)).copy()
        c = layer.cache(T)
        return out, c.expert_of.copy(), c.perm_token.copy(), c.gate_of.copy(), layer.losses()

    def same(a, b):
        return all(np.array_equal(np.asarray(u).view(np.uint8), np.asarray(v).view(np.uint8)) for u, v in zip(a, b))

    layer.forward_device(xb.ptr, T, ob.ptr)
    plain = snapshot()
    ob.upload(np.zeros_like(x))
    kt = layer.forward_kernel_times(xb.ptr, T, ob.ptr)
    assert same(snapshot(), plain)
    decode = "decode" in layer.kernel_name()   # decode-shaped: the combine rides in the down launch
    assert kt["gate_up"] > 0 and kt["down"] > 0 and (kt["combine"] > 0) != decode and kt["empty"] == 0
    assert abs(kt["total"] - sum(v for k, v in kt.items() if k != "total")) <= 1e-6
    assert kt["total"] < 5.0          # milliseconds: these are kernel durations, not garbage
    if shape["shared"] if "shared" in shape else False:
        assert kt["shared"] > 0 or "decode" in layer.kernel_name()   # decode-shaped: the shared expert rides in the product launches
    ob.upload(np.zeros_like(x))
    st = layer.forward_timed(xb.ptr, T, ob.ptr)
    assert same(snapshot(), plain) and st["total"] > 0
    # one stage again, by itself
    for stage in ("gate_up", "down", "combine"):
        ob.upload(np.zeros_like(x))
        layer.forward_device(xb.ptr, T, ob.ptr)
        ms = layer.replay_stage(stage, 5)
        if stage == "combine" and decode:
            assert ms is None
            continue
        assert ms is not None and 0 < ms < 5.0
        assert layer.enqueue_stage(stage, 2)
        assert same(snapshot(), plain), stage
    front = layer.kernel_name().startswith("mfma_bf16_decode_front")
    assert front == (T <= 32 and shape["d"] * shape["F"] < 100_000)
    assert (layer.replay_stage("router", 2) is None) == front   # the routing has no launch of its own there
    assert (layer.replay_stage("dispatch", 2) is None) == ("decode" in layer.kernel_name())
    assert layer.replay_stage("empty", 2) is None
    layer.close()
    xb.free()
    ob.free()


@pytest.mark.parametrize("act,E,inside", [("bf16", 8, True), ("f32", 8, True), ("bf16", 6, False)])
def test_kernel_times_are_those_of_the_calls_own_launches(device, act, E, inside):
    """A gate/up launch that does the dispatch's work does it here too: no time for a launch that the call does not have (six
    experts: it has one)."""
    t = synth.make(small_workload(seed=92, act=act, wt=act, d=64, E=E, k=2, F=64, T=300))
    layer = gpu_layer(device, t)
    x = synth.f32_to_bf16_bits(t.x) if act == "bf16" else t.x
    xb, ob = DeviceBuffer(device, x.nbytes).upload(x), DeviceBuffer(device, x.nbytes)
    kt = layer.forward_kernel_times(xb.ptr, 300, ob.ptr)
    assert (kt["dispatch"] == 0) == inside and min(kt["router"], kt["gate_up"], kt["down"], kt["combine"]) > 0
    assert layer.forward_timed(xb.ptr, 300, ob.ptr)["dispatch"] > 0
    layer.close()
    xb.free()
    ob.free()


@pytest.mark.parametrize("act,wt,shape,parts", [
    ("bf16", "bf16", dict(d=64, E=4, k=2, F=1408, T=40, shared_d_ff=1408), 4),
    ("bf16", "int8", dict(d=768, E=8, k=2, F=1408, T=90, shared_d_ff=2112), 2),
    ("f32", "int8", dict(d=128, E=4, k=1, F=1472, T=120, shared_d_ff=1472), 4),     # products over a bf16 copy of the rows
    ("f32", "f32", dict(d=64, E=4, k=2, F=704, T=33, shared_d_ff=704), 4),
    ("f32", "bf16", dict(d=512, E=4, k=2, F=352, T=33, shared_d_ff=352), 4),
])
def test_timed_forwards_share_a_reduction_out_as_the_call_does(device, act, wt, shape, parts):
    """The shared expert rides in the call's own launches and has launches of its own in the timed ones; the parts of the reduction
    are the same in both, and in the replay of the down product, which is the routed experts' alone.  Bits are, too, where the rows
    are bf16; over f32 rows a launch of fewer tiles may sum in another order (1e-6: some roundings of 2^-24)."""
    t = synth.make(small_workload(seed=93, act=act, wt=wt, shared=True, **shape))
    T = shape["T"]
    layer = gpu_layer(device, t, max_tokens=8 * T)
    x = synth.f32_to_bf16_bits(t.x) if act == "bf16" else t.x
    xb, ob = DeviceBuffer(device, x.nbytes).upload(x), DeviceBuffer(device, x.nbytes)

    def output():
        device.synchronize()
        return ob.download(np.empty_like(x)).copy()

    def same(a, b):
        return rel_l2(a, b) <= 1e-6 if wt == act == "f32" or shape["F"] == 352 else np.array_equal(a.view(np.uint8), b.view(np.uint8))

    layer.forward_device(xb.ptr, T, ob.ptr)
    plain = output()
    assert last_products(layer)[1] == parts
    for measured in (layer.forward_timed, layer.forward_kernel_times):
        ob.upload(np.zeros_like(x))
        assert measured(xb.ptr, T, ob.ptr)["shared"] > 0
        assert last_products(layer)[1] == parts and same(output(), plain)
    layer.forward_device(xb.ptr, T, ob.ptr)
    rows = layer.expert_rows(int(layer.cache(T).offsets[-1]))[1]
    assert layer.enqueue_stage("down", 1) and layer.enqueue_stage("combine", 1)
    assert same(output(), plain) and same(layer.expert_rows(rows.size // shape["d"])[1], rows)
    layer.close()
    xb.free()
    ob.free()
