"""Host matrices through the pinned pool: results in pinned blocks, pageable ones, a pool that is given back to, rows
longer than one piece of the copy, f32 rows of bf16 layers rounded by the library."""
import ctypes as C
import subprocess
import sys
import threading

import numpy as np
import pytest

from conftest import ROOT
from helpers import gpu_layer, small_workload
from rustingbrain_amd import _lib as L
from rustingbrain_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", ["f32", "bf16"])
@pytest.mark.parametrize("T", [1, 33, 5300])   # results below and above the pinned size, and more than one piece
def test_every_host_entry_point_gives_the_same_bits(device, act, T):
    t = synth.make(small_workload(d=128, E=4, k=2, F=64, T=T, seed=81, act=act, wt="bf16"))
    x = t.x.copy()
    x[0, :3] = [np.nan, np.inf, np.float32(1.00390625)]   # conversions: NaN, infinity, a tie between two bf16 values
    layer = gpu_layer(device, t)
    out, cache = layer.forward_train(x)
    plain = np.ascontiguousarray(synth.f32_to_bf16_bits(x) if act == "bf16" else x)
    res = np.empty_like(plain)
    lib = L.load()
    assert lib.rbmoe_forward_host(layer.handle, plain.ctypes.data, T, 128, None, None, None, res.ctypes.data) == L.OK
    want = synth.bf16_bits_to_f32(res).reshape(T, 128) if act == "bf16" else res
    assert np.array_equal(out.view(np.uint32), want.view(np.uint32))
    again = layer.cache(T)
    for name in ("expert_of", "counts", "offsets", "perm_slot", "perm_token"):
        assert np.array_equal(getattr(cache, name), getattr(again, name)), name
    assert np.array_equal(cache.probabilities.view(np.uint32), again.probabilities.view(np.uint32))
    assert cache.assignments[2:] == again.assignments[2:]   # (the first row is all NaN)
    layer.close()


def test_blocks_go_back_to_the_pool_and_exhausting_it_is_harmless(device):
    lib = L.load()
    a = device.empty((1 << 20,), np.float32)
    at = a.ctypes.data
    view = a[5:]
    del a
    assert device.empty((1 << 20,), np.float32).ctypes.data != at   # still in use through the view
    del view
    assert device.empty((1 << 20,), np.float32).ctypes.data == at   # kept for the next one of its size
    p = C.c_void_p()
    assert lib.rbmoe_host_alloc(device.handle, (1 << 30) + 1, C.byref(p)) == L.OUT_OF_MEMORY
    big = device.empty(((1 << 28) + 1,), np.float32)                 # above the pool's bound: ordinary memory
    assert big.size == (1 << 28) + 1
    del big
    t = synth.make(small_workload(d=64, E=4, k=2, F=64, T=40, seed=82))
    layer = gpu_layer(device, t)
    want, _ = layer.forward_train(t.x)
    held = device.empty(((1 << 30) - (64 << 20),), np.uint8)
    blocks = [held] + [device.empty((8 << 20,), np.uint8) for _ in range(10)]   # nothing pinned is left for the rest
    rows = np.tile(t.x, (1, 1))
    got, _ = layer.forward_train(rows)
    assert np.array_equal(got, want)
    del blocks, held
    layer.close()


def test_threads_take_and_give_blocks_at_once(device):
    errors = []

    def work(seed):
        rng = np.random.default_rng(seed)
        for _ in range(200):
            a = device.empty((int(rng.integers(5000, 200000)),), np.float32)
            a[:] = seed
            if a[0] != seed or a[-1] != seed or a.sum() != np.float32(seed) * a.size:
                errors.append(seed)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    [th.start() for th in threads]
    [th.join() for th in threads]
    assert not errors


def test_blocks_outliving_the_last_context_are_not_kept():
    """In a process of its own: this one's contexts live on."""
    code = """
import ctypes as C
import subprocess
import sys
import numpy as np
import rustingbrain_amd as rb
from rustingbrain_amd import _lib as L
def pool():
    used, kept = C.c_uint64(), C.c_uint64()
    assert L.load().rbmoe_internal_host_pool(C.byref(used), C.byref(kept)) == L.OK
    return used.value, kept.value
dev = rb.Device.open(0)
a, b = dev.empty((1 << 20,), np.float32), dev.empty((1 << 20,), np.float32)
del b
assert pool() == (4 << 20, 4 << 20), pool()
dev.close()
assert pool() == (4 << 20, 0), pool()   # what was kept is gone, what is in use is not
a[:] = 1
del a
assert pool() == (0, 0), pool()
dev = rb.Device.open(0)
c = dev.empty((1 << 20,), np.float32)
del c
assert pool() == (0, 4 << 20), pool()
dev.close()
assert pool() == (0, 0), pool()
print("pool ok")
"""
    done = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert done.returncode == 0 and "pool ok" in done.stdout, done.stderr[-2000:]


@pytest.mark.parametrize("T", [40, 9000])   # tables in ordinary memory, and in pinned blocks
def test_a_table_that_is_kept_keeps_no_other_table(device, T):
    t = synth.make(small_workload(d=64, E=8, k=2, F=64, T=T, seed=84))
    layer = gpu_layer(device, t)
    _, cache = layer.forward_train(t.x)

    def memory(a):
        while isinstance(a.base, np.ndarray):
            a = a.base
        return a.ctypes.data, a.ctypes.data + a.nbytes

    names = ("expert_of", "gate_of", "counts", "offsets", "perm_slot", "perm_token", "probabilities", "log_sum_exp")
    spans = sorted(memory(getattr(cache, n)) for n in names)
    assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))
    for n in names:
        lo, hi = memory(getattr(cache, n))
        assert hi - lo <= 4 * max(T * 8, 9)   # a table's own bytes
    layer.close()
