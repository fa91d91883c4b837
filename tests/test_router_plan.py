"""How a large-batch call is routed is decided once, from the pointers its launch gets: which kernel takes the rows depends
on their alignment, and the kernels' blocks - what the dispatch launch counts by - differ in tokens."""
import ctypes as C

import pytest

from rustingbrain_amd import _lib as L

ALIGNED = 1 << 21
TOKENS = (1, 9, 40, 203, 2048, 2049, 4096, 4097, 8192, 8193, 16384)


def plan(d, E, k, T, bf16, norm, quantized, fused, x):
    fn = L.load().rbmoe_internal_router_plan
    fn.restype = C.c_int
    fn.argtypes = [C.c_int32] * 8 + [C.c_uint64, C.POINTER(C.c_int32)]
    out = (C.c_int32 * 4)()
    assert fn(d, E, k, T, bf16, norm, quantized, fused, x, out) == L.OK
    return tuple(out)


def router_slice(d, E, k, T, bf16, norm, quantized):
    fn = L.load().rbmoe_internal_router_slice
    fn.restype = C.c_int
    fn.argtypes = [C.c_int32] * 7
    return fn(d, E, k, T, bf16, norm, quantized)


@pytest.mark.parametrize("quantized", [0, 1])
@pytest.mark.parametrize("norm", [0, 1])
@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("offset", [0, 2, 4, 8, 14])
def test_the_launch_takes_the_plan_the_dispatch_counts_by(offset, bf16, norm, quantized):
    for d, E, k in ((768, 16, 2), (512, 8, 2), (1024, 64, 6), (768, 5, 1), (320, 12, 3), (1024, 33, 2), (33, 6, 2), (40, 80, 2)):
        for T in TOKENS:
            for fused in (0, 1):
                block, apart, taken, again = plan(d, E, k, T, bf16, norm, quantized, fused, ALIGNED + offset)
                case = (d, E, k, T, fused)
                assert taken == 1, case
                assert again == block, case   # the stage by itself writes the blocks the dispatch's own replay counts by
                if norm and offset:
                    # the normed rows are the layer's own: planned like a call whose rows they are
                    assert apart == 1 and block == plan(d, E, k, T, bf16, 0, quantized, fused, ALIGNED)[0], case


def test_small_blocks_serve_calls_that_would_not_fill_the_chip():
    assert [plan(768, 16, 2, T, 1, 0, 0, 1, ALIGNED)[0] for T in (40, 203, 2048, 2049, 4096, 4097)] == [8, 8, 8, 16, 16, 32]
    assert plan(768, 16, 2, 203, 1, 0, 0, 1, ALIGNED + 2)[0] == 32   # rows off a 16-byte boundary without a norm in front


def test_experts_of_a_block_are_shared_out_to_at_most_one_round_of_workgroups():
    assert [router_slice(512, 64, 2, T, 1, 0, 0) for T in (5, 256, 257, 512, 513, 1020, 1024)] == [8, 8, 16, 16, 32, 32, 32]
    assert [router_slice(512, E, 2, 40, 1, 0, 0) for E in (8, 31, 32, 33, 44)] == [0, 0, 8, 8, 8]
    assert [router_slice(d, 32, 2, 40, 1, 0, 0) for d in (256, 504, 512, 544, 1024)] == [0, 0, 8, 8, 8]
    assert router_slice(512, 64, 2, 2048, 1, 0, 0) == 0   # a round of workgroups as it is
