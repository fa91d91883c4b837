"""The weighted sum of a token's expert rows (combine_vec_kernel): slots of every count it is compiled for and one short of it, rows of
whole waves of pieces and others, padded tokens - bit for bit the sum of the expert rows that the layer itself reports, one rounded
product and one rounded addition a slot in ascending position."""
import numpy as np
import pytest

import rustingbrain_amd as rb
from helpers import gpu_layer, small_workload
from rustingbrain_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", range(1, 9))
@pytest.mark.parametrize("d,act,wt", [(512, "bf16", "bf16"), (768, "bf16", "bf16"), (1024, "bf16", "int8"), (64, "f32", "f32"),
                                      (256, "f32", "f32"), (320, "f32", "bf16"), (768, "f32", "bf16")])
def test_sum_of_expert_rows(device, d, act, wt, k):
    T = 131
    t = synth.make(small_workload(d=d, E=16, k=k, F=64, T=T, seed=41 + k, act=act, wt=wt))
    layer = gpu_layer(device, t)
    valid = np.arange(T) % 5 != 3
    out, cache = layer.forward_train(t.x, rb.Layout(valid=valid))
    routed = int(cache.offsets[-1])
    _, y = layer.expert_rows(routed)
    want = np.zeros((T, d), np.float32)
    gates = np.asarray(cache.gate_of, np.float32).reshape(-1)
    for pos, slot in enumerate(np.asarray(cache.perm_slot)[:routed]):
        want[slot // k] += gates[slot] * y[pos]
    if act == "bf16":
        want = synth.round_bf16(want)
    assert routed == int(valid.sum()) * k and not out[~valid].any()
    np.testing.assert_array_equal(out, want)
    layer.close()
