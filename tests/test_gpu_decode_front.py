"""The routing beside the gate/up products (at most 32 tokens): every combination of row type, weights, router and norm
that the launch has a variant for, several routing workgroups, a k past the combine's first slots, ragged teams."""
from types import SimpleNamespace

import numpy as np
import pytest

from conftest import rel_l2
from helpers import assert_routing_identical, gpu_layer, oracle_layer, small_workload
from oracle import rb_oracle as orc
from rustingbrain_amd import Layout, synth
from rustingbrain_amd import _lib as L

pytestmark = pytest.mark.gpu

SHAPES = [
    dict(d=128, E=4, k=2, F=64, T=1, shared=True, shared_d_ff=192),     # untouched experts, sides of different widths
    dict(d=192, E=8, k=2, F=320, T=9),                                  # two routing workgroups, an odd block count
    dict(d=768, E=8, k=5, F=64, T=32, shared=True, shared_d_ff=64),     # full tiles, five slots a token
    dict(d=1024, E=64, k=8, F=64, T=31),                                # router rows in groups, eight slots a token
]


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("act,wt,q8", [("bf16", "bf16", False), ("bf16", "int8", False), ("bf16", "int8", True),
                                       ("f32", "bf16", False), ("f32", "int8", True)])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "d{d}_E{E}_k{k}_F{F}_T{T}".format(**s))
def test_matches_the_oracle(device, shape, act, wt, q8, norm):
    t = synth.make(small_workload(seed=95, act=act, wt=wt, **shape))
    T, d, E = shape["T"], shape["d"], shape["E"]
    layer, ref_layer = gpu_layer(device, t), oracle_layer(t)
    if q8:
        ref_layer.router_q, ref_layer.router_s = synth.quantize_rows(t.router)
        layer.set_router_q8(ref_layer.router_q, ref_layer.router_s)
    valid = (np.arange(T) % 5 != 3).astype(np.uint8)
    bias = synth.normal((E,), 0.5, 95, 98)
    rows = t.x
    if norm:
        w = (1.0 + 0.1 * synth.normal((d,), 1.0, 95, 97)).astype(np.float32)
        layer.set_feed_forward_norm(w, 1e-6)
        rows = orc.rmsnorm(t.x, w, 1e-6)
        if act == "bf16":
            rows = synth.round_bf16(rows)
    ref = ref_layer.forward(rows, valid=valid, router_bias=bias, threads=4)
    layout = Layout(valid=[bool(v) for v in valid])
    call = layer.forward_block if norm else layer.forward_train
    for _ in range(2):   # twice: the arrival counters are back at zero
        out, cache = call(t.x, layout, router_bias=bias)
        assert layer.kernel_name().startswith("mfma_bf16_decode")
        assert_routing_identical(cache, ref)
        assert rel_l2(out, ref.out + t.x if norm else ref.out) <= 2e-2
    h, y = layer.expert_rows(int(ref.offsets[-1]))
    assert rel_l2(h, ref.hidden) <= 2e-2 and rel_l2(y, ref.expert_out) <= 2e-2
    assert abs(cache.aux_loss() - ref.aux_loss) <= 1e-6 + 1e-5 * abs(ref.aux_loss)
    layer.close()


@pytest.mark.parametrize("act,wt", [("bf16", "bf16"), ("f32", "int8")])
def test_block_step_with_the_fused_router_switched_off(device, act, wt):
    """RBMOE_OPT_FUSED_ROUTER 0 speaks of the large-batch routing: a decode step still norms its rows on the way."""
    t = synth.make(small_workload(d=64, E=6, k=2, F=64, T=9, seed=71, act=act, wt=wt))
    layer = gpu_layer(device, t)
    layer.set_feed_forward_norm((1.0 + 0.1 * synth.normal((64,), 1.0, 71, 97)).astype(np.float32), 1e-6)
    out, cache = layer.forward_block(t.x)
    layer.forward_block(t.x[::-1].copy())   # (what the layer's buffers hold afterwards is another call's)
    layer.set_option(L.OPT_FUSED_ROUTER, 0)
    again, cache_again = layer.forward_block(t.x)
    assert_routing_identical(cache_again, SimpleNamespace(**{**vars(cache), "lse": cache.log_sum_exp}))
    assert np.array_equal(again, out)
    layer.close()
