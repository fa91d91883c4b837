"""Counts, offsets, positions, tile table and losses of calls with many router blocks: expert counts around the four columns
of a workgroup and the 64 of a wave, parts with no block, with a few and with more than are kept in registers."""
import numpy as np
import pytest

import rustingbrain_amd as rb
from conftest import rel_l2
from helpers import assert_routing_identical, gpu_layer, oracle_layer, small_workload
from rustingbrain_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,k,T", [(256, 2, 545), (255, 1, 1999), (65, 2, 2081), (64, 6, 2049), (63, 3, 9000), (7, 2, 18753)])
def test_layout_of_many_router_blocks(device, E, k, T):
    t = synth.make(small_workload(seed=61, act="bf16", wt="bf16", d=64, E=E, k=k, F=64, T=T))
    valid = (np.arange(T) % 17 != 4).astype(np.uint8)
    bias = np.zeros(E, np.float32)
    bias[E - 1] = -50  # an expert nobody picks
    ref = oracle_layer(t).forward(t.x, valid=valid, router_bias=bias, threads=8)
    layer = gpu_layer(device, t)
    out, cache = layer.forward_train(t.x, rb.Layout(valid=[bool(v) for v in valid]), router_bias=bias)
    assert_routing_identical(cache, ref)
    # f32 sums of at most T probabilities in another order
    assert abs(cache.aux_loss() - ref.aux_loss) <= 1e-5 * abs(ref.aux_loss)
    assert abs(cache.z_loss() - ref.z_loss) <= 1e-5 * abs(ref.z_loss)
    assert rel_l2(out, ref.out) <= 1e-2
    layer.close()
