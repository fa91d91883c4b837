"""Expert widths between two multiples of a matrix-core tile: the kernels see them rounded up with zero rows and
columns, callers see their own widths (outputs, hidden rows, gradients).  Not where the rows are f32 and the weights are
not: the matrix cores would take them as bf16, so such layers keep the any-shape kernels and f32 accuracy."""
import numpy as np
import pytest

from conftest import rel_l2
from helpers import assert_routing_identical, gpu_layer, oracle_layer, small_workload
from rustingbrain_amd import synth
from test_gpu_backward import check_backward

pytestmark = pytest.mark.gpu

# (the mixed layers' 1e-5 is what test_gpu_backward_any.py holds them to)
# one column past a tile, one short of it, the default model's 352, a quarter of a tile (the smallest that is rounded)
WIDTHS = [(65, 63), (352, 352), (16, 129)]


def mixed(act, wt):
    return act == "f32" and wt != "f32"


@pytest.mark.parametrize("act,wt", [("bf16", "bf16"), ("bf16", "int8"), ("f32", "bf16"), ("f32", "int8"), ("f32", "f32")])
@pytest.mark.parametrize("F,Fs", WIDTHS)
@pytest.mark.parametrize("T", [3, 32, 150])   # separate routing, routing beside the products, large-batch kernels
def test_forward(device, act, wt, F, Fs, T):
    t = synth.make(small_workload(d=64, E=6, k=2, F=F, T=T, seed=61, act=act, wt=wt, shared=True, shared_d_ff=Fs))
    ref = oracle_layer(t).forward(t.x, threads=4)
    layer = gpu_layer(device, t)
    out, cache = layer.forward_train(t.x)
    assert layer.kernel_name() == "generic" if mixed(act, wt) else layer.kernel_name().startswith("mfma")
    assert_routing_identical(cache, ref)
    tol = 1e-5 if act == "f32" else 2e-2
    assert rel_l2(out, ref.out) <= tol
    h, y = layer.expert_rows(int(ref.offsets[-1]))
    assert rel_l2(h, ref.hidden) <= tol and rel_l2(y, ref.expert_out) <= tol
    layer.close()


@pytest.mark.parametrize("act,wt", [("bf16", "bf16"), ("f32", "bf16"), ("f32", "f32")])
@pytest.mark.parametrize("F,Fs", WIDTHS[:2])
def test_backward(device, act, wt, F, Fs):
    t = synth.make(small_workload(d=64, E=5, k=2, F=F, T=150, seed=62, act=act, wt=wt, shared=True, shared_d_ff=Fs))
    layer, _, _ = check_backward(device, t, tol=1e-5 if act == "f32" else None)
    assert layer.kernel_name() == "generic" if mixed(act, wt) else layer.kernel_name().startswith("mfma")
    layer.close()
