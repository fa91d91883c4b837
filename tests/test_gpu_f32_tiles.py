"""Products over f32 rows at the sizes where a tile, a slice of the reduction or the way of the operands into LDS changes,
and values that three bf16 parts do not hold."""
import time

import numpy as np
import pytest

from bench import DeviceBuffer
from conftest import rel_l2
from helpers import assert_routing_identical, gpu_layer, oracle_layer, small_workload
from rustingbrain_amd import synth
from test_gpu_row_pointers import run

pytestmark = pytest.mark.gpu

# One row up to several 64-row tiles an expert; widths of whole slices (64, 192), of half slices (96), of no whole pieces
# (70, 37), a last tile of one feature (257) and more features than fit one round of small tiles (1408)
SHAPES = [dict(d=64, E=4, k=2, F=192, T=1), dict(d=128, E=3, k=1, F=96, T=97), dict(d=96, E=4, k=2, F=257, T=65),
          dict(d=70, E=5, k=2, F=37, T=40), dict(d=512, E=8, k=2, F=1408, T=130), dict(d=512, E=8, k=2, F=1408, T=515),
          dict(d=256, E=3, k=2, F=682, T=1030), dict(d=192, E=2, k=2, F=1408, T=1500)]


# 1e-5 is f32's: a chain of 1408 rounded additions is off by at most 1408 * 2^-24 = 8e-5 of the sum of magnitudes, and by its
# root, 2e-6, on average; the mixed layers of test_gpu_ragged_widths.py are held to the same
@pytest.mark.parametrize("wt", ["f32", "bf16", "int8"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "d{d}_F{F}_T{T}".format(**s))
def test_tiles(device, shape, wt):
    if wt != "f32" and shape["F"] % 64 == 0 and shape["d"] % 64 == 0:
        shape = {**shape, "F": shape["F"] + 32}   # (such a layer's rows would be rounded to bf16)
    t = synth.make(small_workload(seed=71, act="f32", wt=wt, shared=True, shared_d_ff=shape["F"], **shape))
    ref = oracle_layer(t).forward(t.x, threads=8)
    layer = gpu_layer(device, t)
    out, cache = layer.forward_train(t.x)
    assert_routing_identical(cache, ref)
    h, y = layer.expert_rows(int(ref.offsets[-1]))
    assert rel_l2(h, ref.hidden) <= 1e-5 and rel_l2(y, ref.expert_out) <= 1e-5
    assert rel_l2(out, ref.out) <= 1e-5
    layer.close()


@pytest.mark.parametrize("T", [1, 150])
@pytest.mark.parametrize("wt", ["bf16", "int8"])
def test_rows_off_a_piece(device, wt, T):
    """Rows of whole 16-byte pieces that do not start on one travel element by element."""
    t = synth.make(small_workload(d=64, E=4, k=2, F=96, T=T, seed=73, act="f32", wt=wt))
    layer = gpu_layer(device, t)
    got, _, _ = run(device, layer, np.ascontiguousarray(t.x), 4, lambda x, o: layer.forward_device(x, T, o))
    assert rel_l2(got.view(np.float32).reshape(T, 64), oracle_layer(t).forward(t.x, threads=4).out) <= 1e-5
    layer.close()


@pytest.mark.parametrize("T", [20, 300])
@pytest.mark.parametrize("wt,F", [("f32", 64), ("f32", 45), ("bf16", 96), ("int8", 45)])
def test_values_that_do_not_split(device, wt, F, T):
    """Infinities, values within a rounding of the largest, NaN and subnormal values in the rows, infinities in f32 weights:
    the hidden rows hold infinities and NaN where f32 arithmetic on the values themselves puts them."""
    t = synth.make(small_workload(d=64, E=3, k=2, F=F, T=T, seed=72, act="f32", wt=wt))
    x = t.x
    x[1, 5], x[2, 9], x[3, 60] = np.inf, -np.inf, np.nan
    x[4, 0], x[5, 63] = 3.4e38, -3.4e38        # rounded to bf16 these are infinities
    x[6], x[7] = 1e-41, x[7] * 1e-36           # subnormal values, and values whose parts are
    if wt == "f32":
        t.experts[1]["gate"][3, 7] = np.inf
        t.experts[2]["up"][0, 0] = -np.inf
    with np.errstate(all="ignore"):
        ref = oracle_layer(t).forward(x, threads=4)
    layer = gpu_layer(device, t)
    layer.forward_train(x)
    R = int(ref.offsets[-1])
    h, _ = layer.expert_rows(R)
    want = np.asarray(ref.hidden[:R])
    np.testing.assert_array_equal(np.isnan(h), np.isnan(want))
    np.testing.assert_array_equal(np.where(np.isinf(h), h, 0), np.where(np.isinf(want), want, 0))
    ok = np.isfinite(want) & (np.abs(want) < 1e30)
    assert np.isinf(want).any() and np.isnan(want).any() and ok.any()
    assert rel_l2(h[ok], want[ok]) <= 1e-5
    layer.close()


@pytest.mark.parametrize("T", [1, 40, 300])
@pytest.mark.parametrize("wt,F", [("f32", 64), ("f32", 45), ("bf16", 96), ("int8", 45)])
def test_products_next_to_the_largest_value(device, wt, F, T):
    """x w is within f32, the product of the nearest bf16 values of both is not: the hidden rows are finite, as the oracle's."""
    v, w = (1.99 * 2.0 ** 126, 2 * 1.004) if wt == "f32" else (2.0 ** 127 * (1 - 2.0 ** -10), 2.0)
    v, w = np.float32(v), np.float32(w)
    assert np.isfinite(v * w)
    with np.errstate(over="ignore"):
        assert np.isinf(np.float32(synth.round_bf16(np.array([v]))[0] * synth.round_bf16(np.array([w]))[0]))
    t = synth.make(small_workload(d=64, E=3, k=1, F=F, T=T, seed=75, act="f32", wt=wt))
    t.router[:, 0] = 0
    for e in t.experts:
        gate, up = (e["gate_q"], e["up_q"]) if wt == "int8" else (e["gate"], e["up"])
        gate[::3], up[::3] = 0, 0
        gate[::3, 0], up[::3, 1] = w, 1
        gate[1::3, 0] = 0   # (what else they multiply stays as it is)
        gate[2::3, 0] = 0
        up[1::3, 0] = 0
        up[2::3, 0] = 0
        if wt == "int8":
            e["gate_s"][:], e["up_s"][:] = 1, 1
    t.x[:, 0], t.x[:, 1] = v, np.float32(2.0 ** -3)
    ref = oracle_layer(t).forward(t.x, threads=4)
    layer = gpu_layer(device, t)
    layer.forward_train(t.x)
    h, _ = layer.expert_rows(T)
    want = np.asarray(ref.hidden[:T])
    assert np.isfinite(want).all() and (np.abs(want[:, ::3]) > 4e37).all()
    assert np.isfinite(h).all()
    np.testing.assert_allclose(h[:, ::3], want[:, ::3], rtol=2.0 ** -22)   # one product, one halving
    rest = np.arange(F) % 3 != 0
    assert rel_l2(h[:, rest], want[:, rest]) <= 1e-5
    layer.close()


# A product is off by 2^-24 of itself; each of a row's K terms next to the smallest value is rounded to a multiple of 2^-149.
# Rows of 2^-122 in three bf16 parts, the last of which would be below 2^-133, are off by 1e-4.
SCALES = [80, 89, 91, 100, 108, 112, 118, 122]


def assert_rows_close(got, want, K):
    got, want = got.astype(np.float64), want.astype(np.float64)
    err, size = np.sqrt(((got - want) ** 2).mean(axis=1)), np.sqrt((want ** 2).mean(axis=1))
    assert (size > 0).all()
    np.testing.assert_array_less(err, 1e-5 * size + K * 2.0 ** -150)


@pytest.mark.parametrize("T", [8, 40, 300])
@pytest.mark.parametrize("wt,F", [("f32", 64), ("f32", 45), ("bf16", 96), ("int8", 45)])
def test_rows_of_tiny_values(device, wt, F, T):
    """Tiny sums over rows that hold a large value too, and rows of nothing but tiny values: each row by itself."""
    t = synth.make(small_workload(d=64, E=3, k=1, F=F, T=T, seed=76, act="f32", wt=wt))
    dense = []
    for e in t.experts:
        if wt == "int8":
            e["up_q"][:, 0] = 0
            m = [e[n + "_q"].astype(np.float64) * e[n + "_s"].astype(np.float64)[:, None] for n in ("gate", "up", "down")]
        else:
            e["up"][:, 0] = 0
            m = [e[n].astype(np.float64) for n in ("gate", "up", "down")]
        dense.append(m)
    t.x[:, 1:] *= np.ldexp(np.float32(1), -np.resize(SCALES, T))[:, None].astype(np.float32)
    t.x[:, 0] = 1
    layer = gpu_layer(device, t)
    _, cache = layer.forward_train(t.x)
    h, y = layer.expert_rows(T)
    tok = np.asarray(cache.perm_token[:T])
    x = t.x[tok].astype(np.float64)
    expert = np.asarray(cache.expert_of).reshape(-1)[tok]
    for e, (gate, up, down) in enumerate(dense):
        of = expert == e
        if not of.any():
            continue
        g = x[of] @ gate.T
        assert_rows_close(h[of], g / (1 + np.exp(-g)) * (x[of] @ up.T), 64)
        assert_rows_close(y[of], h[of].astype(np.float64) @ down.T, F)
    layer.close()


@pytest.mark.parametrize("wt,F,T", [("f32", 64, 40), ("f32", 96, 300), ("bf16", 45, 70)])
def test_gradients_of_tiny_rows(device, wt, F, T):
    """Gradients are proportional to what comes in: rows of 2^-80 to 2^-122 as rows of one."""
    t = synth.make(small_workload(d=64, E=4, k=2, F=F, T=T, seed=77, act="f32", wt=wt))
    layer = gpu_layer(device, t, training=True, aux_w=0, z_w=0)
    gout = np.random.default_rng(5).standard_normal(t.x.shape).astype(np.float32)
    scale = np.ldexp(np.float32(1), -np.resize(SCALES, T))[:, None].astype(np.float32)
    layer.forward_train(t.x)
    whole = layer.backward(gout).astype(np.float64)
    tiny = layer.backward(gout * scale)
    assert_rows_close(tiny, whole * scale, 64 + 2 * F)
    layer.close()


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("wt,F", [("f32", 704), ("bf16", 352), ("int8", 352)])
def test_sums_taken_again_cost_little_and_leave_the_neighbours_alone(device, wt, F, value):
    """Sums that are not numbers are taken again on the f32 matrix unit.  A sixteenth of the bf16 unit's rate by three or six
    products is at most five times the products' time; one lane at a time it was thirty times that of the whole call."""
    T = 1024
    t = synth.make(small_workload(d=512, E=8, k=2, F=F, T=T, seed=74, act="f32", wt=wt))
    layer = gpu_layer(device, t)
    x = np.ascontiguousarray(t.x)
    some = x.copy()
    some[::7, 100] = value
    outs, times = [], []
    for rows in (x, some, np.full_like(x, value)):
        xb, ob = DeviceBuffer(device, x.nbytes).upload(rows), DeviceBuffer(device, x.nbytes)
        best = 1e9
        for _ in range(6):
            device.synchronize()
            t0 = time.perf_counter()
            for _ in range(10):
                layer.forward_device(xb.ptr, T, ob.ptr)
            device.synchronize()
            best = min(best, time.perf_counter() - t0)
        outs.append(ob.download(np.empty_like(x)).copy())
        times.append(best)
        xb.free()
        ob.free()
    same = np.arange(T) % 7 != 0
    np.testing.assert_array_equal(outs[0][same].view(np.uint32), outs[1][same].view(np.uint32))
    assert not np.isfinite(outs[1][~same]).all(axis=1).any()
    assert max(times[1:]) <= 5 * times[0], times
    layer.close()
