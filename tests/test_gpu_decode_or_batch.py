"""Calls of a few tokens on either side of the lines between the decode-shaped kernels and the large-batch sequence: which
kernels run, and that routing tables and rows are the oracle's on both sides."""
import numpy as np
import pytest

from conftest import rel_l2
from helpers import assert_routing_identical, gpu_layer, oracle_layer, small_workload
from oracle import rb_oracle as orc
from rustingbrain_amd import synth

pytestmark = pytest.mark.gpu

CASES = [  # weights expected to be fetched for nothing beside the routing
    (dict(d=512, E=8, k=2, F=1408, T=1), "mfma_bf16_decode_front"), (dict(d=512, E=16, k=2, F=1408, T=3), "mfma_bf16_decode"),
    (dict(d=512, E=16, k=2, F=1408, T=4), "mfma_bf16_decode_front"), (dict(d=1024, E=32, k=2, F=256, T=9), "mfma_bf16_decode_front"),
    # routing alone in one workgroup: rows that do not fit its LDS, and rows that do
    (dict(d=1024, E=32, k=1, F=640, T=3), "mfma_bf16_decode"), (dict(d=1024, E=32, k=1, F=640, T=4), "mfma_bf16_stream"),
    (dict(d=512, E=32, k=1, F=1408, T=9), "mfma_bf16_decode"), (dict(d=512, E=32, k=1, F=1408, T=10), "mfma_bf16_stream"),
    # routing beside the products: slots and weights
    (dict(d=1024, E=16, k=4, F=704, T=28), "mfma_bf16_decode_front"), (dict(d=1024, E=16, k=4, F=704, T=29), "mfma_bf16_stream")]


@pytest.mark.parametrize("shape,kernel", CASES, ids=lambda s: "d{d}_E{E}_k{k}_F{F}_T{T}".format(**s) if isinstance(s, dict) else s)
def test_few_tokens(device, shape, kernel):
    t = synth.make(small_workload(seed=71, act="bf16", wt="bf16", **shape))
    ref = oracle_layer(t).forward(t.x, threads=8)
    layer = gpu_layer(device, t)
    out, cache = layer.forward_train(t.x)
    assert layer.kernel_name() == kernel
    assert_routing_identical(cache, ref)
    assert rel_l2(out, ref.out) <= 1e-2  # bf16 hidden and expert rows: 2^-9 a rounding, a few in a row
    layer.close()


@pytest.mark.parametrize("shape,kernel", [
    (dict(d=512, E=8, k=2, F=1408, T=1), "mfma_bf16_decode_front"), (dict(d=512, E=16, k=2, F=1408, T=4), "mfma_bf16_decode"),
    (dict(d=1024, E=32, k=2, F=512, T=3), "mfma_bf16_decode_front"), (dict(d=1024, E=32, k=2, F=768, T=3), "mfma_bf16_decode")],
    ids=lambda s: "d{d}_E{E}_k{k}_F{F}_T{T}".format(**s) if isinstance(s, dict) else s)
def test_few_tokens_behind_a_norm(device, shape, kernel):
    """Every workgroup of the combined launch norms the rows again, so its line lies lower for a block step."""
    t = synth.make(small_workload(seed=72, act="bf16", wt="bf16", **shape))
    w = (1.0 + 0.1 * synth.normal((shape["d"],), 1.0, 72, 97)).astype(np.float32)
    rows = orc.rmsnorm(t.x, w, 1e-6)
    ref = oracle_layer(t).forward(synth.round_bf16(rows), threads=8)
    layer = gpu_layer(device, t)
    layer.set_feed_forward_norm(w, 1e-6)
    out, cache = layer.forward_block(t.x)
    assert layer.kernel_name() == kernel
    assert_routing_identical(cache, ref)
    assert rel_l2(out, ref.out + t.x) <= 1e-2
    layer.close()
