"""bf16 rows routed on the f32 matrix cores (route_exact_kernel, and the routing beside the decode-shaped products): blocks of 8,
16 and 32 tokens at their edges, steps that fill no block of 16, experts that fill no round of 16 and several groups of router
rows, both routers - and rows and router weights whose products are not exact, which take the sums one rounding at a time.
Everything the router leaves is the oracle's bit for bit."""
import numpy as np
import pytest

import rustingbrain_amd as rb
from helpers import assert_routing_identical, gpu_layer, oracle_layer, small_workload
from oracle import rb_oracle as orc
from rustingbrain_amd import synth
from test_router_plan import ALIGNED, plan, routes_on_matrix_cores, rows_launch

pytestmark = pytest.mark.gpu

SHAPES = [dict(d=64, E=4, k=2, T=1), dict(d=192, E=17, k=2, T=9), dict(d=320, E=16, k=1, T=47), dict(d=64, E=15, k=3, T=2063),
          dict(d=704, E=8, k=2, T=2065), dict(d=192, E=33, k=2, T=4129), dict(d=1024, E=48, k=2, T=2100)]
OFF_QUANTIZED = [s for s in SHAPES if s["E"] == 33]   # (short rows under a quantized router of many experts: other kernels)
FORMS = ["plain", "range", "tiny", "huge", "infinite", "f32 router", "tiny router"]
# (a quantized router holds whole numbers)
FORMS_AND_ROUTERS = [(form, quantized) for form in FORMS for quantized in (False, True) if not (quantized and "router" in form)]


def shape_id(s):
    return "d{d}_E{E}_k{k}_T{T}".format(**s)


def rows_and_router(t, form):
    x, router = t.x.copy(), t.router.copy()
    rows = slice(x.shape[0] // 2, None)          # (the first blocks stay on the matrix cores)
    if form == "one in a block":                 # ... and a row or two of each of the others leave them
        x[rows.start::29, 7] = 2.0 ** -80
    elif form == "range":                          # the least and the greatest magnitudes that stay there, and zeros
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
    return x, router


def layers(device, t, router, quantized):
    layer, oracle = gpu_layer(device, t), oracle_layer(t)
    oracle.router = router
    if quantized:
        q, s = synth.quantize_rows(router)
        layer.set_router_q8(q, s)
        oracle.router_q, oracle.router_s = q, s
    else:
        layer.set_router(router)
    return layer, oracle


@pytest.mark.parametrize("form,quantized", FORMS_AND_ROUTERS)
@pytest.mark.parametrize("shape", SHAPES, ids=shape_id)
def test_routing_of_bf16_rows(device, shape, form, quantized):
    t = synth.make(small_workload(F=64, seed=37, act="bf16", wt="int8", **shape))
    x, router = rows_and_router(t, form)
    layer, oracle = layers(device, t, router, quantized)
    # (up to 32 tokens the routing runs beside the products, by the same body)
    assert shape["T"] <= 32 or routes_on_matrix_cores(**shape, quantized=quantized) != (quantized and shape in OFF_QUANTIZED)
    with np.errstate(all="ignore"):
        ref = oracle.forward(x, threads=8)
    _, cache = layer.forward_train(x, rb.Layout())
    assert_routing_identical(cache, ref)
    layer.close()


# Calls of more than 16 experts in several rounds of workgroups and of more than 256 K pairs, and rounds of 16 and of 8 experts whose
# router rows follow one another into the same place.
LARGE = [(dict(d=64, E=64, k=2, T=4200), False), (dict(d=256, E=33, k=3, T=9000), False), (dict(d=1280, E=40, k=2, T=2100), False),
         (dict(d=1024, E=48, k=2, T=8200), False), (dict(d=1024, E=48, k=2, T=8190), True), (dict(d=1536, E=40, k=2, T=2100), True),
         (dict(d=512, E=25, k=2, T=14340), True), (dict(d=2048, E=64, k=2, T=300), True)]


@pytest.mark.parametrize("form", ["plain", "one in a block", "tiny"])
@pytest.mark.parametrize("shape,quantized", LARGE, ids=lambda s: shape_id(s) if isinstance(s, dict) else str(s))
def test_large_calls(device, shape, quantized, form):
    assert routes_on_matrix_cores(**shape, quantized=quantized)
    t = synth.make(small_workload(F=64, seed=39, act="bf16", wt="int8", **shape))
    x, router = rows_and_router(t, form)
    layer, oracle = layers(device, t, router, quantized)
    T, E = shape["T"], shape["E"]
    valid = np.arange(T) % 7 != 3
    bias = synth.normal((E,), 0.5, 39, 98)
    ref = oracle.forward(x, valid=valid.astype(np.uint8), router_bias=bias, threads=8)
    _, cache = layer.forward_train(x, rb.Layout(valid=valid), router_bias=bias)
    assert_routing_identical(cache, ref)
    if form == "plain":   # behind a norm, in the launch or in front of it
        w = (1.0 + 0.1 * synth.normal((shape["d"],), 1.0, 39, 97)).astype(np.float32)
        layer.set_feed_forward_norm(w, 1e-6)
        ref = oracle.forward(synth.round_bf16(orc.rmsnorm(x, w, 1e-6)), threads=8)
        _, cache = layer.forward_block(x)
        assert_routing_identical(cache, ref)
    layer.close()


# Several rounds of workgroups two of which lie on a compute unit: blocks of 32 with fewer router rows, and blocks of 16.
TWO_A_UNIT = [(dict(d=512, E=33, k=2, T=8225), False, 32), (dict(d=768, E=24, k=3, T=8193), False, 16),
              (dict(d=1024, E=64, k=6, T=8193), False, 16), (dict(d=512, E=48, k=2, T=15001), True, 16)]


@pytest.mark.parametrize("form", ["plain", "one in a block"])
@pytest.mark.parametrize("shape,quantized,tokens", TWO_A_UNIT, ids=lambda s: shape_id(s) if isinstance(s, dict) else str(s))
def test_two_workgroups_a_unit(device, shape, quantized, tokens, form):
    assert plan(shape["d"], shape["E"], shape["k"], shape["T"], 1, 0, int(quantized), 1, ALIGNED, 1)[0] == tokens
    test_large_calls(device, shape, quantized, form)


@pytest.mark.parametrize("shape,quantized,tokens", TWO_A_UNIT, ids=lambda s: shape_id(s) if isinstance(s, dict) else str(s))
def test_room_for_two_workgroups_a_unit(shape, quantized, tokens):
    EG, block, lds = rows_launch(shape["d"], shape["E"], shape["k"], shape["T"], bf16=1, quantized=int(quantized), exact=1)
    assert EG > 0 and block == tokens and 2 * lds <= 160 * 1024


@pytest.mark.parametrize("shape,quantized", [(dict(d=1024, E=64, k=2, T=4200), False), (dict(d=1024, E=48, k=2, T=8190), True)])
@pytest.mark.parametrize("which", ["one", "all"])
def test_rows_out_of_range_do_not_hold_up_the_others(device, which, shape, quantized):
    """One tiny element in one row, and one in every row.  A row's exact sums are 2 x E x 1024 operations on the vector units instead of
    the matrix cores: times the routing without any, 1.5 and 3.6 (quantized 1.3 and 2.7), and 16.5 to 18.7 where one element holds up its
    block's sums, one after the other.  The line lies as many times above the former as below the latter."""
    assert routes_on_matrix_cores(**shape, quantized=quantized)
    t = synth.make(small_workload(F=64, seed=38, act="bf16", wt="int8", **shape))
    layer = gpu_layer(device, t)
    if quantized:
        layer.set_router_q8(*synth.quantize_rows(t.router))

    def routing(x):
        layer.forward_train(x)
        return min(layer.replay_stage("router", 10) for _ in range(3))

    plain = routing(t.x)
    x = t.x.copy()
    x[:1 if which == "one" else None, 3] = synth.round_bf16(np.full(1, 1e-30, np.float32))
    assert routing(x) < 8 * plain
    layer.close()
