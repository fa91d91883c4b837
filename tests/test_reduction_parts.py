"""Where a matrix-core call's down product is shared out over workgroups: on either side of the lines that were measured."""
import ctypes as C

import pytest

from rustingbrain_amd import _lib as L


def stream_parts(T, E, k, F, Fs, d, int8):
    fn = L.load().rbmoe_internal_stream_parts
    fn.restype = C.c_int
    fn.argtypes = [C.c_int32] * 7
    return fn(T, E, k, F, Fs, d, int8)


@pytest.mark.parametrize("d,E,k,F,Fs,T,bf16,int8", [
    # long reductions of few rows: quarters, and halves where the rows are more
    (768, 8, 2, 2752, 0, 100, 2, 4), (512, 8, 1, 2752, 0, 186, 4, 4), (768, 8, 2, 1408, 0, 83, 1, 4), (768, 8, 2, 1408, 0, 200, 1, 2),
    (256, 4, 2, 1792, 0, 60, 4, 4), (768, 8, 2, 2752, 2752, 200, 2, 4),
    # short ones, or a shared expert's rows beside them: no gain, or a loss
    (768, 4, 4, 1088, 0, 64, 1, 1), (256, 4, 2, 1088, 1088, 186, 1, 4), (768, 8, 2, 1408, 1408, 186, 1, 2), (512, 16, 4, 1088, 0, 150, 1, 1),
    (256, 4, 4, 1408, 1408, 150, 1, 4), (256, 8, 1, 1408, 1408, 600, 1, 4),
    # under a thousand columns, over 64 tiles, over half a million elements
    (512, 8, 2, 960, 0, 60, 1, 1), (768, 24, 1, 2752, 0, 60, 1, 1), (512, 8, 2, 2752, 0, 513, 1, 1),
])
def test_where_reductions_are_shared_out(d, E, k, F, Fs, T, bf16, int8):
    assert (stream_parts(T, E, k, F, Fs, d, 0), stream_parts(T, E, k, F, Fs, d, 1)) == (bf16, int8)
