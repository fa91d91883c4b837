"""A quantized router's products where they take a launch of their own: one turn of the 32 column lanes, several slices, a
rest off the lanes, rows off 16 bytes, more than 64 experts, launches of few and of many workgroups, and a router
that goes from int8 back to f32 - against the oracle bit for bit."""
import numpy as np
import pytest

import rustingbrain_amd as rb
from helpers import assert_routing_identical, gpu_layer, oracle_layer, small_workload
from oracle import rb_oracle as orc
from rustingbrain_amd import synth

pytestmark = pytest.mark.gpu

SHAPES = [dict(d=32, E=72, k=2, T=1), dict(d=40, E=72, k=2, T=65), dict(d=31, E=65, k=1, T=64), dict(d=392, E=64, k=2, T=3000),
          dict(d=100, E=64, k=1, T=4161), dict(d=288, E=64, k=1, T=4161), dict(d=136, E=9, k=2, T=20000)]


@pytest.mark.parametrize("act", ["bf16", "f32"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "d{d}_E{E}_k{k}_T{T}".format(**s))
def test_products_of_a_quantized_router(device, shape, act):
    t = synth.make(small_workload(seed=71, act=act, wt="int8", F=32, **shape))
    layer, oracle = gpu_layer(device, t), oracle_layer(t)
    bias = np.linspace(-0.2, 0.2, shape["E"]).astype(np.float32)
    q, s = orc.q8_quantize(t.router, 1)
    for quantized in (True, False):
        oracle.router_q, oracle.router_s = (q, s) if quantized else (None, None)
        if quantized:
            layer.set_router_q8(q, s)
        else:
            layer.set_router(t.router)
        ref = oracle.forward(t.x, router_bias=bias, threads=8)
        _, cache = layer.forward_train(t.x, rb.Layout(), router_bias=bias)
        assert_routing_identical(cache, ref)
    layer.close()
