"""Grouped products in tiles of 160 rows (large calls of many tiles), against the oracle: last tiles of one to five token blocks, last
feature tiles of at most 64 features, a shared expert in the launches, f32 rows."""
import ctypes as C

import numpy as np
import pytest

import rustingbrain_amd as rb
from conftest import rel_l2
from helpers import assert_routing_identical, gpu_layer, last_products, oracle_layer, small_workload
from rustingbrain_amd import _lib as L
from rustingbrain_amd import synth


def tile_rows(rows, E, F, d):
    fn = L.load().rbmoe_internal_stream_tile
    fn.restype = C.c_int
    fn.argtypes = [C.c_int32] * 4
    return fn(rows, E, F, d)


def test_where_tiles_are_tall():
    # (routed rows, experts, width, d): both sides of the smallest size, and where whole tiles a compute unit speak for either
    assert [tile_rows(*c) for c in ((7650, 8, 1408, 1024), (12000, 8, 1408, 768), (20000, 8, 1408, 768), (32768, 8, 1408, 768),
                                    (98304, 64, 704, 1024), (0, 8, 1408, 768))] == [128, 160, 128, 160, 160, 128]


def test_tiles_are_not_tall_for_a_gain_of_less_than_2_percent():
    assert [tile_rows(*c) for c in ((16800, 8, 1408, 768), (21200, 16, 704, 1024), (36000, 64, 704, 1024))] == [128, 128, 128]


CASES = [
    ("bf16", "bf16", dict(d=320, E=48, k=4, F=960, T=3500)),                                    # half a last feature tile
    ("bf16", "int8", dict(d=320, E=48, k=4, F=960, T=3500)),
    ("f32", "int8", dict(d=256, E=64, k=4, F=704, T=7300)),
    ("bf16", "bf16", dict(d=768, E=48, k=8, F=1088, T=1000, shared=True, shared_d_ff=192)),     # a shared expert in the launches
    ("f32", "bf16", dict(d=576, E=9, k=2, F=960, T=6000, shared=True, shared_d_ff=64)),         # ... and in launches of its own
]


@pytest.mark.gpu
@pytest.mark.parametrize("act,wt,shape", CASES, ids=lambda s: "d{d}_E{E}_k{k}_F{F}_T{T}".format(**s) if isinstance(s, dict) else s)
def test_products(device, act, wt, shape):
    d, E, k, F, T = (shape[n] for n in ("d", "E", "k", "F", "T"))
    assert tile_rows(T * k, E, F, d) == 160
    t = synth.make(small_workload(seed=57, act=act, wt=wt, **shape))
    bias = synth.normal((E,), 0.3, 57, 98)   # groups of all sizes
    valid = (np.arange(T) % 11 != 6).astype(np.uint8)
    ref = oracle_layer(t).forward(t.x, valid=valid, router_bias=bias, threads=8)
    if E > 9:
        assert set(range(5)) <= set(int(-(-(c % 160) // 32)) % 5 for c in ref.counts)   # last tiles of every number of token blocks
    layer = gpu_layer(device, t)
    out, cache = layer.forward_train(t.x, rb.Layout(valid=[bool(v) for v in valid]), router_bias=bias)
    assert_routing_identical(cache, ref)
    h, y = layer.expert_rows(int(ref.offsets[-1]))
    # bf16 operands, f32 sums, one bf16 rounding a row: 2^-9 for the hidden rows, about twice that behind the second product
    assert rel_l2(h, ref.hidden) <= 1e-2
    assert rel_l2(y, ref.expert_out) <= 1e-2
    assert rel_l2(out, ref.out) <= 1e-2
    layer.close()


@pytest.mark.gpu
@pytest.mark.parametrize("padded", [False, True])
@pytest.mark.parametrize("act,wt,shape", CASES, ids=lambda s: "d{d}_E{E}_k{k}_F{F}_T{T}".format(**s) if isinstance(s, dict) else s)
def test_products_with_and_without_padding(device, act, wt, shape, padded):
    d, E, k, F, T = (shape[n] for n in ("d", "E", "k", "F", "T"))
    assert tile_rows(T * k, E, F, d) == 160
    t = synth.make(small_workload(seed=57, act=act, wt=wt, **shape))
    bias = synth.normal((E,), 0.3, 57, 98)   # groups of all sizes
    valid = (np.arange(T) % 11 != 6).astype(np.uint8) if padded else None
    ref = oracle_layer(t).forward(t.x, valid=valid, router_bias=bias, threads=8)
    if E > 9 and not padded:
        assert set(range(5)) <= set(int(-(-(c % 160) // 32)) % 5 for c in ref.counts)   # last tiles of every number of token blocks
    layer = gpu_layer(device, t)
    out, cache = layer.forward_train(t.x, rb.Layout(valid=[bool(v) for v in valid]) if padded else rb.Layout(), router_bias=bias)
    assert last_products(layer)[0] == (128 if padded else 160)   # with padding there are fewer rows than the host knows
    assert_routing_identical(cache, ref)
    h, y = layer.expert_rows(int(ref.offsets[-1]))
    # bf16 operands, f32 sums, one bf16 rounding a row: 2^-9 for the hidden rows, about twice that behind the second product
    assert rel_l2(h, ref.hidden) <= 1e-2
    assert rel_l2(y, ref.expert_out) <= 1e-2
    assert rel_l2(out, ref.out) <= 1e-2
    layer.close()
