"""Where the down product of a large-batch call is shared out over workgroups: on either side of the lines that were measured."""
import ctypes as C

import pytest

from rustingbrain_amd import _lib as L


def parts(T, E, k, F, Fs, d, f32_rows, weight_dtype):
    fn = L.load().rbmoe_internal_parts
    fn.restype = C.c_int
    fn.argtypes = [C.c_int32] * 8
    return fn(T, E, k, F, Fs, d, f32_rows, weight_dtype)


def stream_parts(T, E, k, F, Fs, d, int8):
    return parts(T, E, k, F, Fs, d, 0, L.I8 if int8 else L.BF16)


@pytest.mark.parametrize("int8", [0, 1])
@pytest.mark.parametrize("d,E,k,F,Fs,T,want", [
    # quarters up to 48 tiles and 128 K elements
    (768, 8, 2, 1408, 0, 83, 4), (512, 8, 1, 2752, 0, 186, 4), (256, 4, 2, 1792, 0, 60, 4), (256, 4, 2, 1024, 0, 256, 4), (256, 4, 2, 1024, 0, 257, 2),
    # halves up to 64 tiles and 512 K elements, a shared expert's among them
    (768, 8, 2, 2752, 0, 100, 2), (768, 8, 2, 1408, 0, 200, 2), (768, 8, 2, 2752, 2752, 200, 2), (512, 16, 4, 1088, 0, 150, 2),
    (256, 8, 1, 1408, 1408, 600, 2), (512, 8, 2, 2752, 0, 512, 2),
    # under a thousand columns on either side, over 64 tiles, over half a million elements
    (512, 8, 2, 960, 0, 60, 1), (512, 8, 2, 1408, 960, 60, 1), (768, 24, 1, 2752, 0, 60, 1), (512, 8, 2, 2752, 0, 513, 1),
])
def test_where_reductions_are_shared_out(d, E, k, F, Fs, T, want, int8):
    assert stream_parts(T, E, k, F, Fs, d, int8) == want


# d, experts, a row, width, shared width, rows: while every workgroup has a compute unit to itself, in reductions of at least 288 columns
@pytest.mark.parametrize("wt", [L.F32, L.BF16, L.I8])
@pytest.mark.parametrize("d,E,k,F,Fs,T,want", [
    (64, 4, 2, 1408, 0, 1, 4), (512, 8, 2, 352, 0, 40, 4), (512, 8, 2, 352, 352, 40, 2), (768, 8, 2, 1408, 0, 2, 2), (768, 8, 2, 1408, 0, 16, 1),
    (512, 8, 2, 1408, 0, 1024, 1), (96, 4, 2, 288, 0, 9, 4), (96, 4, 2, 256, 0, 9, 1), (256, 8, 4, 256, 256, 65, 1), (128, 4, 3, 64, 0, 5, 1),
    (96, 4, 2, 352, 256, 9, 1), (96, 4, 2, 350, 0, 9, 1),   # the shorter of the two; no whole slices
])
def test_where_reductions_over_f32_rows_are_shared_out(d, E, k, F, Fs, T, want, wt):
    assert parts(T, E, k, F, Fs, d, 1, wt) == want
