"""The routing launch that keeps a workgroup's whole rows in LDS: 8, 16 and 32 tokens a workgroup, router rows in one
group and in several, both routers, with and without the norm, and the calls at the edges of its rule."""
import numpy as np
import pytest

from conftest import rel_l2
from helpers import assert_routing_identical, gpu_layer, oracle_layer, small_workload
from oracle import rb_oracle as orc
from rustingbrain_amd import Layout, synth
from test_router_plan import ALIGNED, plan, rows_launch

pytestmark = pytest.mark.gpu

SHAPES = [
    dict(d=64, E=5, k=2, T=33),       # 8 tokens a workgroup, the last one short
    dict(d=64, E=16, k=3, T=2049),    # the first call with 16 tokens a workgroup
    dict(d=64, E=9, k=2, T=4097),     # ... and with 32
    dict(d=544, E=9, k=2, T=2049),    # ... rows long enough for the quantized router's 16 tokens
    dict(d=544, E=9, k=2, T=4097),    # ... and 32
    dict(d=544, E=9, k=2, T=8193),    # a second round of workgroups would start: another kernel
    dict(d=1024, E=64, k=6, T=40),    # router rows in groups
    dict(d=1024, E=16, k=2, T=4100),  # 32 tokens do not fit, the norm takes a launch of its own
    dict(d=320, E=12, k=2, T=300),    # lanes of 40 steps (8 lanes) and of 10: a last piece with zeros (32 lanes)
    dict(d=1024, E=33, k=2, T=4200),  # block histograms past the limit of the fused layout scan
]


@pytest.mark.parametrize("act,quantized", [("bf16", False), ("f32", False), ("bf16", True), ("f32", True)])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "d{d}_E{E}_k{k}_T{T}".format(**s))
def test_block_step_routes_like_the_oracle(device, shape, act, quantized):
    t = synth.make(small_workload(F=64, seed=91, act=act, wt="int8" if quantized else "bf16", **shape))
    T, d = shape["T"], shape["d"]
    layer = gpu_layer(device, t)
    ref_layer = oracle_layer(t)
    if quantized:
        q, s = synth.quantize_rows(t.router)
        layer.set_router_q8(q, s)
        ref_layer.router_q, ref_layer.router_s = q, s
    w = (1.0 + 0.1 * synth.normal((d,), 1.0, 91, 97)).astype(np.float32)
    layer.set_feed_forward_norm(w, 1e-6)
    valid = (np.arange(T) % 7 != 3).astype(np.uint8)
    out, cache = layer.forward_block(t.x, Layout(valid=[bool(v) for v in valid]))
    normed = orc.rmsnorm(t.x, w, 1e-6)
    if act == "bf16":
        normed = synth.round_bf16(normed)
    ref = ref_layer.forward(normed, valid=valid, threads=8)
    assert_routing_identical(cache, ref)
    assert rel_l2(out, ref.out + t.x) <= 2e-2
    plain, cache = layer.forward_train(t.x)     # without the norm
    ref = ref_layer.forward(t.x, threads=8)
    assert_routing_identical(cache, ref)
    assert rel_l2(plain, ref.out) <= 2e-2
    assert abs(cache.aux_loss() - ref.aux_loss) <= 1e-5 * abs(ref.aux_loss)
    assert abs(cache.z_loss() - ref.z_loss) <= 1e-5 * abs(ref.z_loss)
    layer.close()


# More than 16 experts over f32 rows, several rounds of workgroups: blocks of 32, 16 and 8 tokens, the last one short, router rows in
# one group and in several, and the line behind which route_fused_kernel keeps long rows.
ROUNDS = [(dict(d=256, E=33, k=2, T=8225), False, 32), (dict(d=512, E=32, k=2, T=8195), False, 16),
          (dict(d=1024, E=64, k=6, T=4201), False, 8), (dict(d=1024, E=40, k=2, T=4111), True, 8),
          (dict(d=512, E=17, k=2, T=8200), False, 32), (dict(d=776, E=24, k=2, T=8200), False, 32)]


@pytest.mark.parametrize("shape,quantized,tokens", ROUNDS, ids=lambda s: "d{d}_E{E}_k{k}_T{T}".format(**s) if isinstance(s, dict) else str(s))
def test_several_rounds_over_f32_rows(device, shape, quantized, tokens):
    assert plan(shape["d"], shape["E"], shape["k"], shape["T"], 0, 0, int(quantized), 1, ALIGNED)[0] == tokens
    test_block_step_routes_like_the_oracle(device, shape, "f32", quantized)


# More than 16 experts over f32 rows: (router rows in LDS together, tokens a block) in several rounds of workgroups, the last block short,
# router rows in one group and in several, blocks that were halved and not; and one round where route_fused_kernel does not have the rows.
ROWS_IN_LDS = [(dict(d=256, E=33, k=2, T=8225), False, (33, 32)), (dict(d=512, E=32, k=2, T=8195), False, (20, 16)),
               (dict(d=1024, E=64, k=6, T=4201), False, (10, 8)), (dict(d=1024, E=40, k=2, T=4111), True, (8, 8)),
               (dict(d=512, E=28, k=2, T=8200), False, (20, 16)), (dict(d=512, E=24, k=2, T=10925), False, (20, 16)),
               (dict(d=512, E=40, k=2, T=12291), False, (40, 32)), (dict(d=64, E=20, k=2, T=13111), False, (20, 32)),
               (dict(d=128, E=28, k=2, T=4201), False, (28, 32)), (dict(d=768, E=20, k=2, T=10243), True, (12, 32)),
               # not taken: route_fused_kernel has the rows
               (dict(d=512, E=17, k=2, T=8200), False, (0, 0)), (dict(d=776, E=24, k=2, T=8200), False, (0, 0)),
               (dict(d=768, E=20, k=2, T=8200), True, (0, 0))]


@pytest.mark.parametrize("shape,quantized,want", ROWS_IN_LDS, ids=lambda s: "d{d}_E{E}_k{k}_T{T}".format(**s) if isinstance(s, dict) else str(s))
def test_f32_rows_in_lds(device, shape, quantized, want):
    assert rows_launch(shape["d"], shape["E"], shape["k"], shape["T"], quantized=int(quantized))[:2] == want
    test_block_step_routes_like_the_oracle(device, shape, "f32", quantized)
