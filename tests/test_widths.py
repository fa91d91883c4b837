"""Which expert widths a layer's kernels see, and that rounding them refuses no layer that its true widths would allow."""
import ctypes as C

import pytest

from rustingbrain_amd import MoeConfig
from rustingbrain_amd import _lib as L

ANY, BF16_CORES, F32_CORES = 0, 1, 2


def widths(d, F, act, wt, Fs=0, T=64, E=8, k=2, training=False):
    cfg = MoeConfig.new(E, k, F).with_shared_expert(Fs > 0)._c(d, act, wt, T, Fs)
    fn = L.load().rbmoe_internal_widths
    fn.restype = C.c_int
    fn.argtypes = [C.POINTER(L.Config), C.c_int32, C.POINTER(C.c_int32)]
    out = (C.c_int32 * 3)()
    rc = fn(C.byref(cfg), int(training), out)
    return tuple(out) if rc == L.OK else rc


@pytest.mark.parametrize("act,wt,F,Fs,want", [
    ("bf16", "bf16", 352, 352, (384, 384, BF16_CORES)), ("bf16", "int8", 65, 63, (128, 64, BF16_CORES)),
    ("bf16", "bf16", 16, 0, (64, 64, BF16_CORES)), ("bf16", "bf16", 15, 0, (15, 15, ANY)),   # four times the work, and more
    ("f32", "f32", 341, 0, (352, 352, F32_CORES)), ("f32", "f32", 15, 0, (15, 15, ANY)),
    ("f32", "bf16", 384, 0, (384, 384, BF16_CORES)), ("f32", "bf16", 352, 0, (352, 352, ANY)),
    ("f32", "bf16", 341, 910, (352, 928, ANY)), ("f32", "int8", 17, 15, (32, 15, ANY)),   # whole slices up to twice the work
    ("f32", "int8", 384, 352, (384, 352, ANY)), ("bf16", "f32", 384, 0, (384, 384, ANY)),
])
def test_widths(act, wt, F, Fs, want):
    assert widths(256, F, act, wt, Fs) == want


def test_a_rounded_width_past_the_backward_products_offsets_is_taken_as_it_is():
    big = dict(act="bf16", wt="bf16", d=64, k=8, T=1 << 20)   # 2^23 rows of 2 x 128 bf16 pre-activations: 4 GiB
    assert widths(F=100, **big) == (128, 128, BF16_CORES)
    assert widths(F=100, training=True, **big) == (100, 100, ANY)
    assert widths(F=128, training=True, **big) == L.UNSUPPORTED   # (nothing was rounded)
    assert widths(F=100, training=True, **{**big, "T": 1 << 19}) == (128, 128, BF16_CORES)
