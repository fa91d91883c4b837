"""The down launch of a row or two (at most four pairs of a row and a side): rows, outputs and tables are those of the launch that
walks the tile table, in every bit."""
import numpy as np
import pytest

import rustingbrain_amd as rb
from conftest import rel_l2
from helpers import assert_routing_identical, gpu_layer, last_products, oracle_layer, small_workload
from rustingbrain_amd import _lib as L
from rustingbrain_amd import synth

pytestmark = pytest.mark.gpu

CASES = [
    dict(d=64, E=4, k=2, F=64, T=1, shared=True, shared_d_ff=192),        # fewer steps than waves; sides of different length
    dict(d=128, E=8, k=2, F=448, T=2, residual=True),                     # two rows, a last wave with less than its share
    dict(d=128, E=4, k=1, F=128, T=4, pad=True),                      # four rows, one of them padding
    dict(d=192, E=6, k=4, F=704, T=1, act="f32", residual=True),          # f32 rows, the most slots
    dict(d=256, E=8, k=2, F=3072, T=1, shared=True, shared_d_ff=1408),    # several batches of steps
    dict(d=64, E=4, k=1, F=64, T=2, shared=True, shared_d_ff=64, pad=True),
    dict(d=64, E=4, k=3, F=64, T=1, pad=True),                            # nothing routed
]


@pytest.mark.parametrize("front", [True, False])
@pytest.mark.parametrize("wt", ["bf16", "int8"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "d{d}_E{E}_k{k}_F{F}_T{T}".format(**c))
def test_gives_the_bits_of_the_tile_table_launch(device, case, wt, front):
    T, k, d = case["T"], case["k"], case["d"]
    t = synth.make(small_workload(d=d, E=case["E"], k=k, F=case["F"], T=T, seed=61, act=case.get("act", "bf16"), wt=wt,
                                  shared=case.get("shared", False), shared_d_ff=case.get("shared_d_ff", 0)))
    valid = np.ones(T, np.uint8)
    if case.get("pad"):
        valid[T // 2] = 0
    residual = synth.round_bf16(synth.normal((T, d), 1.0, 61, 7)) if case.get("residual") else None
    layout = rb.Layout(valid=[bool(v) for v in valid])
    ref = oracle_layer(t).forward(t.x, valid=valid, threads=4)
    R = int(ref.offsets[-1])
    layer = gpu_layer(device, t)
    layer.set_option(L.OPT_DECODE_FRONT, int(front))
    got = []
    for by_expert in (1, 0):
        layer.set_option(L.OPT_DECODE_DOWN_BY_EXPERT, by_expert)
        for _ in range(2):
            out, cache = layer.forward_train(t.x, layout, residual=residual)
            assert ("front" in layer.kernel_name()) == front
            assert_routing_identical(cache, ref)
            got.append((out, layer.expert_rows(R)[1] if R else np.zeros(0, np.float32)))
    for out, rows in got[1:]:
        assert np.array_equal(out.view(np.uint32), got[0][0].view(np.uint32))
        assert np.array_equal(rows.view(np.uint32), got[0][1].view(np.uint32))
    layer.close()


@pytest.mark.parametrize("shape,few", [(dict(k=2, T=2), True), (dict(k=4, T=1), True), (dict(k=3, T=2), False), (dict(k=2, T=3), False),
                                       (dict(k=3, T=1, shared=True), True), (dict(k=4, T=1, shared=True), False),
                                       (dict(k=1, T=2, shared=True), True)])
def test_up_to_four_pairs_of_a_row_and_a_side(device, shape, few):
    t = synth.make(small_workload(d=128, E=8, F=64, seed=62, act="bf16", wt="bf16", **shape))
    layer = gpu_layer(device, t)
    out, _ = layer.forward_train(t.x)
    assert "decode" in layer.kernel_name() and last_products(layer)[2] == few
    assert rel_l2(out, oracle_layer(t).forward(t.x, threads=4).out) <= 1e-2
    layer.close()


@pytest.mark.parametrize("front", [True, False])
@pytest.mark.parametrize("wt", ["bf16", "int8"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "d{d}_E{E}_k{k}_F{F}_T{T}".format(**c))
def test_the_launch_of_a_row_or_two_runs(device, case, wt, front):
    t = synth.make(small_workload(d=case["d"], E=case["E"], k=case["k"], F=case["F"], T=case["T"], seed=61, act=case.get("act", "bf16"), wt=wt,
                                  shared=case.get("shared", False), shared_d_ff=case.get("shared_d_ff", 0)))
    layer = gpu_layer(device, t)
    layer.set_option(L.OPT_DECODE_FRONT, int(front))
    for by_expert in (1, 0):
        layer.set_option(L.OPT_DECODE_DOWN_BY_EXPERT, by_expert)
        layer.forward_train(t.x)
        # (int8 weights behind a routing launch of its own stay with the tile table)
        assert last_products(layer)[2] == (by_expert == 1 and (front or wt == "bf16"))
    layer.close()
