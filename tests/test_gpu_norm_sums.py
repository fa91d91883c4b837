"""The norm in front of the layer over rows whose sum of squares is hard to take out of order: the routing follows the normed
rows in every bit, so a sum off by one rounding anywhere shows.  Widths that divide among a wave's lanes and one that does not;
row counts of one decode launch, of its longer form, of every size of routing block and of a norm in a launch of its own."""
import numpy as np
import pytest

from helpers import gpu_layer, oracle_layer, small_workload
from rustingbrain_amd import synth

pytestmark = pytest.mark.gpu


def rows(rng, T, d):
    x = rng.standard_normal((T, d)).astype(np.float32)
    kinds = [
        lambda: np.full(d, rng.choice([1.0, 1.5, 3.0])),              # every sum exact, then a tie a step
        lambda: 2.0 ** rng.integers(-12, 13, d),                      # ties of either parity
        lambda: np.where(np.arange(d) < d - d // 4, 0.0, rng.standard_normal(d)),   # the sum starts late
        lambda: rng.standard_normal(d) * 1e-20,                       # subnormal squares
        lambda: rng.standard_normal(d) * 2.0 ** np.linspace(-30, 30, d),            # a power of two passed at every step
        lambda: np.where(np.arange(d) == 0, 4096.0, rng.standard_normal(d) * 0.01),  # additions of less than a unit
        lambda: rng.standard_normal(d) * 1e18,                        # sums near the largest, some past it
        lambda: np.where(np.arange(d) == d // 2, np.inf, rng.standard_normal(d)),
        lambda: np.where(np.arange(d) == d - 1, np.nan, rng.standard_normal(d)),
        lambda: np.zeros(d),
    ]
    for i in range(T):
        if i % 16 < len(kinds):
            x[i] = kinds[(i + T) % len(kinds)]()
    return x


@pytest.mark.parametrize("act,wt,T", [("bf16", "bf16", 1), ("f32", "bf16", 8), ("bf16", "int8", 9), ("bf16", "bf16", 32),
                                      ("f32", "f32", 203), ("bf16", "bf16", 2100), ("f32", "int8", 4100), ("bf16", "bf16", 8300)])
@pytest.mark.parametrize("d", [256, 320, 512, 768, 1024])
def test_sums_are_the_references(device, d, act, wt, T):
    t = synth.make(small_workload(d=d, E=4, k=2, F=64, T=T, seed=d + T, act=act, wt=wt))
    rng = np.random.default_rng(T)
    x = rows(rng, T, d) if T > 1 else (rng.standard_normal((1, d)) * 2.0 ** np.linspace(-30, 30, d)).astype(np.float32)
    rounder = synth.round_bf16 if act == "bf16" else None
    x = rounder(x) if rounder else x
    nw = rng.uniform(0.5, 1.5, d).astype(np.float32)
    layer = gpu_layer(device, t)
    layer.set_feed_forward_norm(nw, 1e-6)
    with np.errstate(all="ignore"):
        _, _, ref = oracle_layer(t).forward_block(x, nw, 1e-6, round_normed=rounder, threads=8)
    _, cache = layer.forward_block(x)
    got, want = cache.probabilities, ref.probabilities
    assert np.isnan(want).any() == (T > 1)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    whole = ~np.isnan(want)
    np.testing.assert_array_equal(got[whole].view(np.uint32), want[whole].view(np.uint32))
    np.testing.assert_array_equal(cache.expert_of, ref.expert_of)
    layer.close()
