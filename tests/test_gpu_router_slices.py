"""A few tokens by many experts: a block's experts shared out over workgroups, the last of which goes on with all of them.
Slices of 8, 16 and 32 experts, a last slice that is shorter, blocks with remainders, a norm, f32 rows beside their bf16
copy, padding, a bias; called again and again (the arrival counters return to zero), against the oracle bit for bit."""
import numpy as np
import pytest

import rustingbrain_amd as rb
from conftest import rel_l2
from helpers import assert_routing_identical, gpu_layer, oracle_layer, small_workload
from oracle import rb_oracle as orc
from rustingbrain_amd import synth
from test_router_plan import router_slice

pytestmark = pytest.mark.gpu

# (experts, choices, tokens) -> experts of a workgroup
SHAPES = [dict(E=64, k=6, T=33, n=8), dict(E=64, k=2, T=256, n=8), dict(E=64, k=2, T=257, n=16), dict(E=64, k=4, T=1020, n=32),
          dict(E=32, k=4, T=40, n=8), dict(E=32, k=1, T=512, n=8), dict(E=32, k=2, T=513, n=16), dict(E=44, k=3, T=77, n=8),
          dict(E=33, k=2, T=41, n=8), dict(E=44, k=3, T=1020, n=32), dict(E=40, k=2, T=420, n=16)]
# 512 columns: a wave takes the norm of a row; 544 (17 steps of 32 columns): a thread does
CASES = [(512, s) for s in SHAPES] + [(544, SHAPES[i]) for i in (0, 2, 3, 9)]


@pytest.mark.parametrize("act,wt,quantized", [("bf16", "bf16", False), ("f32", "bf16", False), ("f32", "f32", False), ("bf16", "int8", True)])
@pytest.mark.parametrize("d,shape", CASES, ids=["d{}_E{E}_k{k}_T{T}".format(d, **s) for d, s in CASES])
def test_experts_of_a_block_shared_out(device, d, shape, act, wt, quantized):
    shape = dict(shape)
    slice_ = shape.pop("n")
    for norm in (0, 1):
        if not (norm and quantized):
            assert router_slice(d, shape["E"], shape["k"], shape["T"], act == "bf16", norm, quantized) == slice_
    t = synth.make(small_workload(seed=67, act=act, wt=wt, d=d, F=64, **shape))
    T, E = shape["T"], shape["E"]
    layer = gpu_layer(device, t)
    oracle = oracle_layer(t)
    if quantized:
        oracle.router_q, oracle.router_s = orc.q8_quantize(t.router, 1)
        layer.set_router_q8(oracle.router_q, oracle.router_s)
    rng = np.random.default_rng(3)
    for turn in range(3):
        valid = (rng.random(T) < (1.0, 0.8, 0.5)[turn]).astype(np.uint8)
        valid[0] = 1
        bias = rng.standard_normal(E).astype(np.float32) if turn else np.zeros(E, np.float32)
        ref = oracle.forward(t.x, valid=valid, router_bias=bias, threads=8)
        _, cache = layer.forward_train(t.x, rb.Layout(valid=[bool(v) for v in valid]), router_bias=bias)
        assert_routing_identical(cache, ref)
    if not quantized:  # behind a norm, which every slice takes and the first one writes out
        nw = rng.uniform(0.5, 1.5, t.x.shape[1]).astype(np.float32)
        layer.set_feed_forward_norm(nw, 1e-6)
        out, _, ref = oracle.forward_block(t.x, nw, 1e-6, round_normed=synth.round_bf16 if act == "bf16" else None, threads=8)
        got, cache = layer.forward_block(t.x)
        assert_routing_identical(cache, ref)
        assert rel_l2(got, out) <= 1e-2
    layer.close()
