"""Gate/up launches whose last feature tile holds at most 64 features: its waves share out the token blocks (three or four of them),
in inference and where the pre-activations are kept, with groups of 1 to 128 rows a tile."""
import numpy as np
import pytest

import rustingbrain_amd as rb
from conftest import rel_l2
from helpers import assert_routing_identical, gpu_layer, oracle_layer, small_workload
from rustingbrain_amd import synth
from test_gpu_backward import check_backward

pytestmark = pytest.mark.gpu


# (over 128 gate/up tiles: launches of fewer have tiles of 64 features)
SHAPES = [dict(d=64, E=70, k=2, F=192, T=3300), dict(d=128, E=72, k=2, F=64, T=7000), dict(d=64, E=32, k=1, F=704, T=2900)]


@pytest.mark.parametrize("wt", ["bf16", "int8"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "d{d}_E{E}_k{k}_F{F}_T{T}".format(**s))
def test_products(device, shape, wt):
    t = synth.make(small_workload(seed=53, act="bf16", wt=wt, shared=True, shared_d_ff=shape["F"] + 128, **shape))
    bias = synth.normal((shape["E"],), 0.3, 53, 98)   # groups of all sizes
    ref = oracle_layer(t).forward(t.x, router_bias=bias, threads=8)
    assert {0, 1, 2, 3} <= set(int(-(-(c % 128) // 32)) % 4 for c in ref.counts)   # last tiles of every number of token blocks
    layer = gpu_layer(device, t)
    out, cache = layer.forward_train(t.x, rb.Layout(), router_bias=bias)
    assert_routing_identical(cache, ref)
    h, y = layer.expert_rows(int(ref.offsets[-1]))
    # bf16 operands, f32 sums, one bf16 rounding a row: 2^-9 for the hidden rows, about twice that behind the second product
    assert rel_l2(h, ref.hidden) <= 1e-2
    assert rel_l2(y, ref.expert_out) <= 1e-2
    assert rel_l2(out, ref.out) <= 1e-2
    layer.close()


def test_pre_activations_are_kept(device):
    check_backward(device, synth.make(small_workload(d=64, E=5, k=2, F=192, T=333, seed=53, act="bf16", wt="bf16")), seed=53)
