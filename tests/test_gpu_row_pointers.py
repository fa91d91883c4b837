"""Device rows that do not start on a 16-byte boundary (any element boundary is a legal pointer): the same bits as from
rows on an allocation's boundary."""
import numpy as np
import pytest

from bench import DeviceBuffer
from conftest import rel_l2
from helpers import gpu_layer, oracle_layer, small_workload
from oracle import rb_oracle as orc
from rustingbrain_amd import _lib as L
from rustingbrain_amd import synth

pytestmark = pytest.mark.gpu


def rows_of(t):
    return synth.f32_to_bf16_bits(t.x) if t.workload.act_dtype == "bf16" else np.ascontiguousarray(t.x, np.float32)


def run(device, layer, rows, offset, call):
    """`call(x, out)` on copies of `rows` that start `offset` bytes behind an allocation's start."""
    x, o = DeviceBuffer(device, rows.nbytes + 64), DeviceBuffer(device, rows.nbytes + 64)
    raw = np.zeros(rows.nbytes + 64, np.uint8)
    raw[offset:offset + rows.nbytes] = rows.view(np.uint8).reshape(-1)
    x.upload(raw)
    o.upload(np.zeros_like(raw))
    call(x.ptr + offset, o.ptr + offset)
    device.synchronize()
    got = o.download(np.empty_like(raw)).copy()
    assert not got[:offset].any() and not got[offset + rows.nbytes:].any()   # nothing written beside the rows
    return got[offset:offset + rows.nbytes], layer.cache(rows.shape[0]), layer.losses()


def same(a, b):
    for f in ("expert_of", "counts", "offsets", "perm_slot", "perm_token", "gate_of", "probabilities", "log_sum_exp"):
        assert np.array_equal(getattr(a[1], f).view(np.uint32), getattr(b[1], f).view(np.uint32)), f
    assert np.array_equal(a[0], b[0])
    # the losses' sums of T positive terms are folded block by block, and another kernel's blocks have other sizes
    for u, v in zip(a[2], b[2]):
        assert abs(u - v) <= len(a[1].log_sum_exp) * 2.0 ** -24 * abs(v)


# rows of 8, 16 and 32 tokens a router block; 40 rows: the smallest that no longer fit one block of 8
@pytest.mark.parametrize("act,wt,quantized", [("bf16", "bf16", False), ("bf16", "int8", True), ("f32", "f32", False),
                                              ("f32", "int8", True)])
@pytest.mark.parametrize("T", [40, 203, 2049, 4097])
def test_block_step(device, T, act, wt, quantized):
    t = synth.make(small_workload(d=64, E=6, k=2, F=64, T=T, seed=17, act=act, wt=wt))
    layer = gpu_layer(device, t)
    ref_layer = oracle_layer(t)
    if quantized:
        q, s = synth.quantize_rows(t.router)
        layer.set_router_q8(q, s)
        ref_layer.router_q, ref_layer.router_s = q, s
    w = (1.0 + 0.1 * synth.normal((64,), 1.0, 17, 97)).astype(np.float32)
    layer.set_feed_forward_norm(w, 1e-6)
    rows = rows_of(t)
    call = lambda x, o: layer.forward_block_device(x, T, o)
    aligned = run(device, layer, rows, 0, call)
    normed = orc.rmsnorm(t.x, w, 1e-6)
    ref = ref_layer.forward(synth.round_bf16(normed) if act == "bf16" else normed, threads=8)
    assert np.array_equal(aligned[1].expert_of, ref.expert_of) and np.array_equal(aligned[1].counts, ref.counts)
    for offset in (4, 8):
        same(run(device, layer, rows, offset, call), aligned)
    layer.close()


@pytest.mark.parametrize("act,wt", [("bf16", "bf16"), ("bf16", "int8"), ("f32", "f32"), ("f32", "bf16")])
@pytest.mark.parametrize("T", [9, 40, 300])
def test_forward(device, T, act, wt):
    t = synth.make(small_workload(d=64, E=6, k=2, F=64, T=T, seed=19, act=act, wt=wt, shared=True, shared_d_ff=128))
    layer = gpu_layer(device, t)
    rows = rows_of(t)
    call = lambda x, o: layer.forward_device(x, T, o)
    aligned = run(device, layer, rows, 0, call)
    for offset in (4, 8):
        got = run(device, layer, rows, offset, call)
        if T > 32:
            same(got, aligned)
        else:   # a few bf16 rows: routed in a launch of their own, the reduction split another way
            assert np.array_equal(got[1].expert_of, aligned[1].expert_of)
            a, b = (synth.bf16_bits_to_f32(r[0].view(np.uint16)) if act == "bf16" else r[0].view(np.float32) for r in (got, aligned))
            assert rel_l2(a, b) <= 5e-3
    layer.close()


@pytest.mark.parametrize("act,wt", [("bf16", "bf16"), ("f32", "f32"), ("f32", "bf16")])
def test_training_step(device, act, wt):
    T = 150
    t = synth.make(small_workload(d=64, E=5, k=2, F=64, T=T, seed=23, act=act, wt=wt, shared=True, shared_d_ff=128))
    layer = gpu_layer(device, t, training=True)
    rows = rows_of(t)
    grad = synth.normal((T, 64), 1.0, 23, 5)
    grad = synth.f32_to_bf16_bits(grad) if act == "bf16" else grad.astype(np.float32)
    results = []
    for offset in (0, 4, 8):
        layer.zero_grads()
        fwd = run(device, layer, rows, offset, lambda x, o: layer.forward_device(x, T, o))
        back = run(device, layer, grad, offset, lambda g, gi: layer.backward_device(g, T, gi))
        grads = [layer.weight_grad(w, 0) for w in (L.W_ROUTER, L.W_GATE, L.W_UP, L.W_DOWN, L.W_SHARED_GATE, L.W_SHARED_UP,
                                                   L.W_SHARED_DOWN)]
        results.append((fwd, back[0], grads))
    for fwd, back, grads in results[1:]:
        same(fwd, results[0][0])
        assert np.array_equal(back, results[0][1])
        assert all(np.array_equal(a, b) for a, b in zip(grads, results[0][2]))
    layer.close()
