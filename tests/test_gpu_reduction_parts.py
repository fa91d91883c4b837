"""Down products whose reduction is shared out over workgroups: in halves and quarters, uneven ones among them, with and without a
shared expert, whatever room the layer has; whole in training and under a memory budget; behind a larger call, and captured."""
import ctypes as C

import numpy as np
import pytest

import rustingbrain_amd as rb
from bench import DeviceBuffer
from conftest import rel_l2
from helpers import assert_routing_identical, gpu_layer, last_products, oracle_layer, small_workload
from rustingbrain_amd import Layout, synth
from test_gpu_graph import Capture
from test_reduction_parts import stream_parts

pytestmark = pytest.mark.gpu

# f32 rows: slices of 64 columns: 22 and 11 in quarters (5 or 6, 2 or 3 each), 3 in halves, 1 whole; of 32 columns (F = 96, 352)
SHAPES = [dict(d=64, E=4, k=2, F=1408, T=1), dict(d=64, E=4, k=4, F=704, T=33), dict(d=128, E=3, k=1, F=192, T=70),
          dict(d=128, E=4, k=3, F=64, T=5), dict(d=96, E=4, k=2, F=96, T=9), dict(d=512, E=8, k=2, F=352, T=40),
          dict(d=512, E=8, k=2, F=1408, T=64)]


# 1e-5: as for the other f32 products (a chain of 1408 rounded additions is off by 2e-6 on average)
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("wt", ["f32", "bf16", "int8"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "d{d}_E{E}_k{k}_F{F}_T{T}".format(**s))
def test_parts(device, shape, wt, shared):
    if wt != "f32" and shape["F"] % 64 == 0 and shape["d"] % 64 == 0:
        shape = {**shape, "F": shape["F"] + 32}   # (such a layer's rows would be rounded to bf16)
    T = shape["T"]
    t = synth.make(small_workload(seed=77, act="f32", wt=wt, shared=shared, shared_d_ff=shape["F"] if shared else 0, **shape))
    valid = (np.arange(T) % 5 != 3).astype(np.uint8)
    residual = synth.normal(t.x.shape, 1.0, 77, 5).astype(np.float32)
    ref = oracle_layer(t).forward(t.x, valid=valid, threads=8)
    for room in (T, T + T // 2 + 1, 2 * T, 8 * T + 3):   # of the layer's rows: whole, halves, quarters
        layer = gpu_layer(device, t, max_tokens=room)
        for _ in range(2):
            out, cache = layer.forward_train(t.x, Layout(valid=[bool(v) for v in valid]), residual=residual)
            assert_routing_identical(cache, ref)
            _, y = layer.expert_rows(int(ref.offsets[-1]))
            assert rel_l2(y, ref.expert_out) <= 1e-5
            assert rel_l2(out, ref.out + residual) <= 1e-5
        layer.close()


# The packed kernels: a reduction of 22 slices of 64 in halves and quarters, of 17 unevenly, the row counts on both sides of the rule's lines
NARROW = [dict(d=64, E=4, k=2, F=1408, T=40), dict(d=512, E=8, k=2, F=1408, T=125), dict(d=512, E=8, k=2, F=1088, T=126),
          dict(d=256, E=3, k=1, F=1024, T=300), dict(d=768, E=8, k=2, F=1408, T=200)]


@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("act,wt", [("bf16", "bf16"), ("bf16", "int8"), ("f32", "bf16"), ("f32", "int8")])
@pytest.mark.parametrize("shape", NARROW, ids=lambda s: "d{d}_E{E}_k{k}_F{F}_T{T}".format(**s))
def test_parts_of_packed_products(device, shape, act, wt, shared):
    T = shape["T"]
    t = synth.make(small_workload(seed=78, act=act, wt=wt, shared=shared, shared_d_ff=shape["F"] if shared else 0, **shape))
    valid = (np.arange(T) % 5 != 3).astype(np.uint8)
    ref = oracle_layer(t).forward(t.x, valid=valid, threads=8)
    got = []
    for room in (T, 2 * T, 4 * T, 8 * T + 3):   # whole rows, as they are rounded; no room for the parts in the first
        layer = gpu_layer(device, t, max_tokens=room)
        for _ in range(2):
            out, cache = layer.forward_train(t.x, Layout(valid=[bool(v) for v in valid]))
            assert_routing_identical(cache, ref)
            _, y = layer.expert_rows(int(ref.offsets[-1]))
            assert rel_l2(y, ref.expert_out) <= 1e-2
            assert rel_l2(out, ref.out) <= 1e-2
        got.append(y)
        layer.close()
    # the same sums in another order, rounded to bf16 once: an element may fall to the neighbouring value now and then
    for y in got[1:]:
        assert rel_l2(y, got[0]) <= 2.0 ** -9


# f32 rows, and the parts without and with a shared expert of the same width: slices of 64 columns: 22, 11 and 5 in quarters (5 or 6, 2 or 3, 1
# or 2 each), 22 in halves, 1 whole; of 32 columns: 9 and 11
PARTS = [(dict(d=64, E=4, k=2, F=1408, T=1), (4, 4)), (dict(d=64, E=4, k=4, F=704, T=33), (4, 4)), (dict(d=128, E=3, k=1, F=320, T=70), (4, 4)),
         (dict(d=128, E=4, k=3, F=64, T=5), (1, 1)), (dict(d=96, E=4, k=2, F=288, T=9), (4, 4)), (dict(d=512, E=8, k=2, F=352, T=40), (4, 2)),
         (dict(d=512, E=8, k=2, F=1408, T=64), (2, 1))]


def shape_id(s):
    return "d{d}_E{E}_k{k}_F{F}_T{T}".format(**s) if isinstance(s, dict) else None


# (1e-5: as above)
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("wt", ["f32", "bf16", "int8"])
@pytest.mark.parametrize("shape,parts", PARTS, ids=shape_id)
def test_parts_whatever_the_layer_has_room_for(device, shape, parts, wt, shared):
    if wt != "f32" and shape["F"] % 64 == 0 and shape["d"] % 64 == 0:
        shape = {**shape, "F": shape["F"] + 32}   # (such a layer's rows would be rounded to bf16)
    T = shape["T"]
    t = synth.make(small_workload(seed=77, act="f32", wt=wt, shared=shared, shared_d_ff=shape["F"] if shared else 0, **shape))
    valid = (np.arange(T) % 5 != 3).astype(np.uint8)
    residual = synth.normal(t.x.shape, 1.0, 77, 5).astype(np.float32)
    ref = oracle_layer(t).forward(t.x, valid=valid, threads=8)
    got = []
    for room in (T, 8 * T + 3):   # of the layer's rows
        layer = gpu_layer(device, t, max_tokens=room)
        for _ in range(2):
            out, cache = layer.forward_train(t.x, Layout(valid=[bool(v) for v in valid]), residual=residual)
            if wt == "f32":
                assert last_products(layer)[1] == parts[shared]
            assert_routing_identical(cache, ref)
            _, y = layer.expert_rows(int(ref.offsets[-1]))
            assert rel_l2(y, ref.expert_out) <= 1e-5
            assert rel_l2(out, ref.out + residual) <= 1e-5
            got.append((out, y, last_products(layer)[1]))
        layer.close()
    for out, y, n in got[1:]:
        assert n == got[0][2] and np.array_equal(out, got[0][0]) and np.array_equal(y, got[0][1])


# The packed kernels: reductions of 15, 17, 22, 29, 33 and 43 slices of 64 in whole, halves and quarters, rows on both sides of the rule's lines
PACKED = [dict(d=64, E=4, k=2, F=1408, T=40), dict(d=512, E=8, k=2, F=1408, T=125), dict(d=768, E=8, k=2, F=1408, T=200),
          dict(d=512, E=8, k=2, F=1088, T=126), dict(d=256, E=3, k=1, F=1856, T=300), dict(d=128, E=8, k=2, F=2112, T=125),
          dict(d=768, E=8, k=2, F=2752, T=140), dict(d=256, E=4, k=2, F=960, T=60)]


@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("act,wt", [("bf16", "bf16"), ("bf16", "int8"), ("f32", "bf16"), ("f32", "int8")])
@pytest.mark.parametrize("shape", PACKED, ids=shape_id)
def test_parts_of_packed_products_whatever_the_layer_has_room_for(device, shape, act, wt, shared):
    d, E, k, F, T = (shape[n] for n in ("d", "E", "k", "F", "T"))
    parts = stream_parts(T, E, k, F, F if shared else 0, d, int(wt == "int8"))
    t = synth.make(small_workload(seed=78, act=act, wt=wt, shared=shared, shared_d_ff=F if shared else 0, **shape))
    valid = (np.arange(T) % 5 != 3).astype(np.uint8)
    ref = oracle_layer(t).forward(t.x, valid=valid, threads=8)
    got = []
    budget = rb.Device.open(0, budget_mib=1 << 16)
    for dev, room, want in ((budget, T, 1), (device, T, parts), (device, 8 * T + 3, parts)):
        layer = gpu_layer(dev, t, max_tokens=room)
        for _ in range(2):
            out, cache = layer.forward_train(t.x, Layout(valid=[bool(v) for v in valid]))
            assert last_products(layer)[1] == want
            assert_routing_identical(cache, ref)
            _, y = layer.expert_rows(int(ref.offsets[-1]))
            assert rel_l2(y, ref.expert_out) <= 1e-2
            assert rel_l2(out, ref.out) <= 1e-2
        got.append((out, y))
        layer.close()
    budget.close()
    # the same sums in another order, rounded to bf16 once: an element may fall to the neighbouring value now and then
    assert rel_l2(got[1][1], got[0][1]) <= 2.0 ** -9
    # whatever the layer has room for
    assert np.array_equal(got[1][0], got[2][0]) and np.array_equal(got[1][1], got[2][1])


def test_the_packed_shapes_take_halves_quarters_and_none():
    took = {stream_parts(s["T"], s["E"], s["k"], s["F"], Fs, s["d"], i) for s in PACKED for Fs in (0, s["F"]) for i in (0, 1)}
    assert took == {1, 2, 4}


def test_a_training_layer_keeps_its_rows_whole(device):
    """Its backward pass reads them."""
    t = synth.make(small_workload(seed=79, act="bf16", wt="bf16", d=64, E=4, k=2, F=1408, T=40))
    layer = gpu_layer(device, t, training=True)
    layer.forward_train(t.x)
    assert last_products(layer)[1] == 1
    layer.close()


@pytest.mark.parametrize("act,wt,F", [("bf16", "int8", 1408), ("f32", "f32", 704)])
@pytest.mark.parametrize("shared", [False, True])
def test_behind_a_larger_call_and_captured(device, act, wt, F, shared):
    """A call in parts leaves nothing to a call in whole and the other way round, eager or replayed from a graph."""
    T, large = 40, 5000
    t = synth.make(small_workload(seed=80, act=act, wt=wt, d=64, E=4, k=2, F=F, T=large, shared=shared, shared_d_ff=F if shared else 0))
    layer = gpu_layer(device, t)
    xh = synth.f32_to_bf16_bits(t.x) if act == "bf16" else t.x
    x = DeviceBuffer(device, xh.nbytes).upload(xh)
    out = DeviceBuffer(device, xh.nbytes)

    def run(rows):
        layer.forward_device(x.ptr, rows, out.ptr)

    def result(rows):
        device.synchronize()
        return out.download(np.empty_like(xh))[:rows].copy()

    run(T)
    small, n = result(T), last_products(layer)[1]
    run(large)
    whole = result(large)
    assert n > 1 and last_products(layer)[1] == 1
    ref = oracle_layer(t).forward(t.x, threads=8)
    assert rel_l2(whole if act == "f32" else synth.bf16_bits_to_f32(whole), ref.out) <= (1e-5 if act == "f32" else 1e-2)
    cap = Capture(C.CDLL("libamdhip64.so"), device, lambda: run(T))
    for _ in range(3):
        cap.replay()
        assert np.array_equal(result(T), small)
        run(large)
        assert np.array_equal(result(large), whole)
    cap.close()
    run(T)
    assert np.array_equal(result(T), small)
    layer.close()
    x.free()
    out.free()
