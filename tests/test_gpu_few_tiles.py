"""Grouped products of launches with few tiles (128-feature workgroups, deep weight ring) and, on the other side of the
line, with enough tiles for the wide ones: reductions of one to seven slices of 64, partial feature tiles, groups of 0 to
129 rows, against the oracle."""
import numpy as np
import pytest

import rustingbrain_amd as rb
from conftest import rel_l2
from helpers import assert_routing_identical, gpu_layer, oracle_layer, small_workload
from rustingbrain_amd import synth

pytestmark = pytest.mark.gpu

SHAPES = [dict(d=64, E=4, k=1, F=64, T=33), dict(d=128, E=3, k=2, F=192, T=129), dict(d=320, E=5, k=2, F=448, T=97),
          dict(d=192, E=8, k=4, F=256, T=257), dict(d=384, E=2, k=1, F=384, T=223),
          # 128 experts: over 128 gate/up and 250 down tiles, so the wide kernel, with the same odd shapes
          dict(d=320, E=128, k=2, F=192, T=260)]


@pytest.mark.parametrize("act,wt", [("bf16", "bf16"), ("bf16", "int8"), ("f32", "bf16")])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "d{d}_E{E}_k{k}_F{F}_T{T}".format(**s))
def test_products_of_few_tiles(device, shape, act, wt):
    t = synth.make(small_workload(seed=51, act=act, wt=wt, shared=True, shared_d_ff=shape["F"] + 64, **shape))
    T, E = shape["T"], shape["E"]
    valid = (np.arange(T) % 13 != 5).astype(np.uint8)
    bias = np.zeros(E, np.float32)
    bias[E - 1] = -50  # an expert nobody picks
    ref = oracle_layer(t).forward(t.x, valid=valid, router_bias=bias, threads=8)
    layer = gpu_layer(device, t)
    out, cache = layer.forward_train(t.x, rb.Layout(valid=[bool(v) for v in valid]), router_bias=bias)
    assert_routing_identical(cache, ref)
    h, y = layer.expert_rows(int(ref.offsets[-1]))
    # bf16 operands, f32 sums, one bf16 rounding a row: 2^-9 for the hidden rows, about twice that behind the second product
    assert rel_l2(h, ref.hidden) <= 1e-2
    assert rel_l2(y, ref.expert_out) <= 1e-2
    assert rel_l2(out, ref.out) <= 1e-2
    layer.close()
