"""How a large-batch call is routed is decided once, from the pointers its launch gets: which kernel takes the rows depends
on their alignment, and the kernels' blocks - what the dispatch launch counts by - differ in tokens."""
import ctypes as C

import pytest

from rustingbrain_amd import _lib as L

ALIGNED = 1 << 21
TOKENS = (1, 9, 40, 203, 2048, 2049, 4096, 4097, 8192, 8193, 16384)


def whole_plan(d, E, k, T, bf16, norm, quantized, exact, fused, x):
    fn = L.load().rbmoe_internal_router_plan
    fn.restype = C.c_int
    fn.argtypes = [C.c_int32] * 9 + [C.c_uint64, C.POINTER(C.c_int32)]
    out = (C.c_int32 * 5)()
    assert fn(d, E, k, T, bf16, norm, quantized, exact, fused, x, out) == L.OK
    return tuple(out)


def plan(d, E, k, T, bf16, norm, quantized, fused, x, exact=0):
    return whole_plan(d, E, k, T, bf16, norm, quantized, exact, fused, x)[:4]


def routes_on_matrix_cores(d, E, k, T, norm=0, quantized=0):
    """Whether bf16 rows are routed by route_exact_kernel, under a router whose weights allow it."""
    return bool(whole_plan(d, E, k, T, 1, norm, quantized, 1, 1, ALIGNED)[4])


def router_slice(d, E, k, T, bf16, norm, quantized, exact=0):
    fn = L.load().rbmoe_internal_router_slice
    fn.restype = C.c_int
    fn.argtypes = [C.c_int32] * 8
    return fn(d, E, k, T, bf16, norm, quantized, exact)


def rows_launch(d, E, k, T, bf16=0, norm=0, quantized=0, exact=0):
    """(router rows in LDS together, tokens of a block, bytes of LDS) of the launch that keeps rows in LDS; zeros where another takes the call."""
    fn = L.load().rbmoe_internal_router_rows
    fn.restype = None
    fn.argtypes = [C.c_int32] * 8 + [C.POINTER(C.c_int32)]
    out = (C.c_int32 * 3)()
    fn(d, E, k, T, bf16, norm, quantized, exact, out)
    return tuple(out)


@pytest.mark.parametrize("exact", [0, 1])
@pytest.mark.parametrize("quantized", [0, 1])
@pytest.mark.parametrize("norm", [0, 1])
@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("offset", [0, 2, 4, 8, 14])
def test_the_launch_takes_the_plan_the_dispatch_counts_by(offset, bf16, norm, quantized, exact):
    for d, E, k in ((768, 16, 2), (512, 8, 2), (1024, 64, 6), (768, 5, 1), (320, 12, 3), (1024, 33, 2), (33, 6, 2), (40, 80, 2)):
        for T in TOKENS:
            for fused in (0, 1):
                block, apart, taken, again = plan(d, E, k, T, bf16, norm, quantized, fused, ALIGNED + offset, exact)
                case = (d, E, k, T, fused)
                assert taken == 1, case
                assert again == block, case   # the stage by itself writes the blocks the dispatch's own replay counts by
                if norm and offset:
                    # the normed rows are the layer's own: planned like a call whose rows they are
                    assert apart == 1 and block == plan(d, E, k, T, bf16, 0, quantized, fused, ALIGNED, exact)[0], case


def test_small_blocks_serve_calls_that_would_not_fill_the_chip():
    assert [plan(768, 16, 2, T, 1, 0, 0, 1, ALIGNED)[0] for T in (40, 203, 2048, 2049, 4096, 4097)] == [8, 8, 8, 16, 16, 32]
    assert [plan(768, 16, 2, T, 1, 0, 0, 1, ALIGNED, 1)[0] for T in (40, 203, 2048, 2049, 4096, 4097)] == [8, 8, 8, 16, 16, 32]
    assert plan(768, 16, 2, 203, 1, 0, 0, 1, ALIGNED + 2)[0] == 32   # rows off a 16-byte boundary without a norm in front


@pytest.mark.parametrize("exact", [0, 1])
def test_experts_of_a_block_are_shared_out_to_at_most_one_round_of_workgroups(exact):
    assert [router_slice(512, 64, 2, T, 1, 0, 0, exact) for T in (5, 256, 257, 512, 513, 1020, 1024)] == [8, 8, 16, 16, 32, 32, 32]
    assert [router_slice(512, E, 2, 40, 1, 0, 0, exact) for E in (8, 31, 32, 33, 44)] == [0, 0, 8, 8, 8]
    assert [router_slice(d, 32, 2, 40, 1, 0, 0, exact) for d in (256, 504, 512, 544, 1024)] == [0, 0, 8, 8, 8]
    assert router_slice(512, 64, 2, 2048, 1, 0, 0, exact) == 0   # a round of workgroups as it is


def test_rows_off_the_matrix_cores():
    """f32 rows and routers whose products are not exact never go there; a norm that a wave does not take does not either."""
    for T in TOKENS:
        for quantized in (0, 1):
            assert whole_plan(768, 16, 2, T, 0, 0, quantized, 1, 1, ALIGNED)[4] == 0
        assert whole_plan(768, 16, 2, T, 1, 0, 0, 0, 1, ALIGNED)[4] == 0
        assert whole_plan(768, 16, 2, T, 1, 0, 0, 1, 0, ALIGNED)[4] == 0
    assert not routes_on_matrix_cores(544, 16, 2, 203, norm=1) and routes_on_matrix_cores(544, 16, 2, 203)


# (d, experts, tokens, quantized): on the matrix cores or not, on either side of each line of the rule
LINES = [
    # up to 16 experts: as many blocks of 32 as lie on the chip together, or a round more where rows are long enough
    (256, 8, 16384, 0, True), (256, 8, 16385, 0, False), (384, 8, 24576, 0, True), (384, 8, 24577, 0, False),
    (512, 8, 16384, 0, True), (512, 8, 16385, 0, False), (768, 16, 8192, 0, True), (768, 16, 8193, 0, False),
    (256, 8, 8192, 1, True), (256, 8, 8193, 1, False), (512, 8, 8193, 1, True), (512, 8, 16384, 1, True), (512, 8, 16385, 1, False),
    # more: any number of rounds
    (256, 17, 9000, 0, True), (1024, 64, 16384, 0, True), (1024, 64, 100000, 0, True), (2048, 64, 16384, 0, True),
    # ... but not with eight tokens a workgroup in many rounds
    (3072, 32, 9600, 0, True), (3072, 32, 9601, 0, False),
    # ... nor under a quantized router with the last round far from full, one round of few workgroups by many experts, short rows
    (512, 32, 14336, 1, True), (512, 32, 14335 - 31, 1, False), (512, 32, 16385, 1, False), (768, 32, 12000, 1, False),
    (768, 32, 24000, 1, True), (1024, 32, 20000, 1, True), (1024, 32, 12000, 1, False), (1024, 24, 16384, 1, False),
    (1280, 32, 9000, 1, False), (1280, 48, 9000, 1, True), (256, 32, 8192, 1, True), (256, 32, 8193, 1, False),
    (512, 48, 5760, 1, True), (512, 48, 5728, 1, False), (128, 17, 8192, 1, False), (128, 16, 8192, 1, True),
]


@pytest.mark.parametrize("d,E,T,quantized,taken", LINES)
def test_where_the_matrix_cores_take_the_rows(d, E, T, quantized, taken):
    assert routes_on_matrix_cores(d, E, 2, T, quantized=quantized) == taken
    if not taken:  # what the rows of any other router get
        assert plan(d, E, 2, T, 1, 0, quantized, 1, ALIGNED, 1) == plan(d, E, 2, T, 1, 0, quantized, 1, ALIGNED, 0)


# f32 rows, (d, experts, tokens, quantized): router rows in LDS together, tokens of a block and whether two workgroups lie on a unit, on either
# side of each line of the rule
F32_ROWS = [
    # up to 16 experts one round of workgroups or two a unit; more in any number of rounds, except where route_fused_kernel has the rows
    (512, 16, 9000, 0, (0, 0, False)), (512, 26, 9000, 0, (0, 0, False)), (512, 27, 9000, 0, (20, 16, True)),
    (512, 24, 10922, 0, (0, 0, False)), (512, 24, 10923, 0, (20, 16, True)),
    (128, 20, 8200, 0, (0, 0, False)), (128, 28, 4200, 0, (28, 32, True)), (64, 24, 16384, 0, (24, 32, True)),
    (768, 24, 10922, 0, (0, 0, False)), (1024, 64, 16384, 0, (10, 8, True)),
    # a quantized router: there too, but not in up to a round and a quarter of workgroups of which a unit takes one
    (640, 24, 8300, 1, (14, 16, True)), (768, 20, 8193, 1, (0, 0, False)), (768, 20, 10240, 1, (0, 0, False)),
    (768, 20, 10241, 1, (12, 32, False)), (768, 30, 8800, 1, (12, 32, False)),
    # two workgroups a unit, unless blocks are halved, router rows taken in twice as many groups and the last round more than half full
    (512, 40, 8192 + 128 * 32, 0, (18, 16, True)), (512, 40, 8193 + 128 * 32, 0, (40, 32, False)), (512, 40, 16384, 0, (40, 32, False)),
    (512, 40, 16385, 0, (18, 16, True)),
    (512, 20, 16384, 0, (20, 16, True)), (1024, 32, 12000, 0, (20, 16, False)), (1024, 32, 13000, 0, (10, 8, True)),
    (1024, 28, 12000, 0, (10, 8, True)),
    (512, 32, 16384, 1, (0, 0, False)), (1024, 32, 16384, 1, (8, 8, True)),
]


@pytest.mark.parametrize("d,E,T,quantized,want", F32_ROWS)
def test_where_f32_rows_lie_in_lds(d, E, T, quantized, want):
    EG, tokens, lds = rows_launch(d, E, 2, T, quantized=quantized)
    assert (EG, tokens, EG > 0 and 2 * lds <= 160 * 1024) == want
