"""bf16 rows routed on the f32 matrix cores (route_exact_kernel, and the routing beside the decode-shaped products): blocks of 8,
16 and 32 tokens at their edges, steps that fill no block of 16, experts that fill no round of 16 and several groups of router
rows, both routers - and rows and router weights whose products are not exact, which take the sums one rounding at a time.
Everything the router leaves is the oracle's bit for bit."""
import numpy as np
import pytest

import rustingbrain_amd as rb
from helpers import assert_routing_identical, gpu_layer, oracle_layer, small_workload
from rustingbrain_amd import synth

pytestmark = pytest.mark.gpu

SHAPES = [dict(d=64, E=4, k=2, T=1), dict(d=192, E=17, k=2, T=9), dict(d=320, E=16, k=1, T=47), dict(d=64, E=15, k=3, T=2063),
          dict(d=704, E=8, k=2, T=2065), dict(d=192, E=33, k=2, T=4129), dict(d=1024, E=48, k=2, T=2100)]
FORMS = ["plain", "range", "tiny", "huge", "infinite", "f32 router", "tiny router"]


@pytest.mark.parametrize("quantized", [False, True])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "d{d}_E{E}_k{k}_T{T}".format(**s))
def test_routing_of_bf16_rows(device, shape, form, quantized):
    if quantized and "router" in form:
        pytest.skip("whole numbers")
    t = synth.make(small_workload(F=64, seed=37, act="bf16", wt="int8", **shape))
    x, router = t.x.copy(), t.router.copy()
    rows = slice(x.shape[0] // 2, None)          # (the first blocks stay on the matrix cores)
    if form == "range":                          # the least and the greatest magnitudes that stay there, and zeros
        x[rows, ::3] = 2.0 ** -72
        x[rows, 1::3] = -(2.0 ** 80 - 2.0 ** 72)
        x[rows, 2::3] = 0.0
    elif form == "tiny":
        x[rows] = synth.round_bf16(x[rows] * np.float32(2.0 ** -100))
    elif form == "huge":
        x[rows] = synth.round_bf16(x[rows] * np.float32(2.0 ** 120))
    elif form == "infinite":
        x[rows, 5] = np.inf
    elif form == "f32 router":
        router += np.float32(1e-5) * synth.normal(router.shape, 1.0, 37, 5)
    elif form == "tiny router":
        router[0, :8] = 2.0 ** -41
    layer, oracle = gpu_layer(device, t), oracle_layer(t)
    oracle.router = router
    if quantized:
        q, s = synth.quantize_rows(router)
        layer.set_router_q8(q, s)
        oracle.router_q, oracle.router_s = q, s
    else:
        layer.set_router(router)
    with np.errstate(all="ignore"):
        ref = oracle.forward(x, threads=8)
    _, cache = layer.forward_train(x, rb.Layout())
    assert_routing_identical(cache, ref)
    layer.close()


@pytest.mark.parametrize("quantized", [False, True])
@pytest.mark.parametrize("which", ["one", "all"])
def test_rows_out_of_range_do_not_hold_up_the_others(device, which, quantized):
    """One tiny element in one row, and one in every row.  A row's exact sums are 2 x 64 x 1024 operations on the vector units instead of
    the matrix cores, a 32nd of a block's for one of its rows: four times the routing's time is far above either, the fifteen that a
    whole block's sums took one after the other are far beyond."""
    t = synth.make(small_workload(d=1024, E=64, k=2, F=64, T=4200, seed=38, act="bf16", wt="int8"))
    layer = gpu_layer(device, t)
    if quantized:
        layer.set_router_q8(*synth.quantize_rows(t.router))

    def routing(x):
        layer.forward_train(x)
        return min(layer.replay_stage("router", 10) for _ in range(3))

    plain = routing(t.x)
    x = t.x.copy()
    x[:1 if which == "one" else None, 3] = synth.round_bf16(np.full(1, 1e-30, np.float32))
    assert routing(x) < 4 * plain
    layer.close()
