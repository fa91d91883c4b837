"""Device rows that do not start on a 16-byte boundary (any element boundary is a legal pointer): the same bits as from
rows on an allocation's boundary."""
import numpy as np
import pytest

from bench import DeviceBuffer
from helpers import gpu_layer, oracle_layer, small_workload
from oracle import rb_oracle as orc
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
    assert np.array_equal(a[0], b[0]) and a[2] == b[2]


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
