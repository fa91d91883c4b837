"""Down products whose reduction is shared out over workgroups: in halves and quarters, uneven ones among them, with and
without a shared expert, in layers with and without room for the parts, and the calls after a captured or larger one."""
import numpy as np
import pytest

from conftest import rel_l2
from helpers import assert_routing_identical, gpu_layer, oracle_layer, small_workload
from rustingbrain_amd import Layout, synth

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
