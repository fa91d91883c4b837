"""Gate/up products that work out their own tiles and write the routing tables on the way, against the oracle's tables and,
bit for bit, against the same call with a dispatch launch (which the timed forward keeps, and a call that writes the gathered
rows out): first and last tile of an expert, experts without rows, a histogram of the largest size, blocks and batches with
remainders, padding, padding only."""
import numpy as np
import pytest
import torch

from helpers import assert_routing_identical, gpu_layer, oracle_layer, small_workload
from rustingbrain_amd import _lib as L
from rustingbrain_amd import synth

pytestmark = pytest.mark.gpu

SHAPES = [dict(E=8, k=2, T=33), dict(E=1, k=1, T=300), dict(E=2, k=2, T=257), dict(E=4, k=1, T=2049), dict(E=16, k=3, T=1000),
          dict(E=32, k=4, T=513), dict(E=64, k=6, T=100), dict(E=64, k=8, T=2048), dict(E=16, k=2, T=8192), dict(E=4, k=2, T=16000),
          dict(E=6, k=2, T=130)]  # (six experts: the dispatch launch)


# widths off 64 (96): rows stay f32 over bf16 and int8 weights too; at 64 those rows are rounded to bf16
@pytest.mark.parametrize("act,wt,shared,F,kernel", [
    ("bf16", "bf16", False, 64, "mfma_bf16_stream"), ("bf16", "int8", True, 64, "mfma_bf16_stream_int8w"),
    ("f32", "bf16", True, 64, "mfma_bf16_stream"), ("f32", "f32", False, 64, "mfma_f32"), ("f32", "f32", True, 64, "mfma_f32"),
    ("f32", "bf16", True, 96, "generic"), ("f32", "int8", True, 96, "generic")])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "E{E}_k{k}_T{T}".format(**s))
def test_tables_and_outputs_without_a_dispatch_launch(device, shape, act, wt, shared, F, kernel):
    t = synth.make(small_workload(seed=61, act=act, wt=wt, shared=shared, shared_d_ff=128 if F == 64 else F, d=64, F=F, **shape))
    T, E = shape["T"], shape["E"]
    dt = torch.bfloat16 if act == "bf16" else torch.float32
    x = torch.from_numpy(np.ascontiguousarray(t.x)).to(dt).cuda()
    bias = np.zeros(E, np.float32)
    if E > 2:
        bias[1], bias[E - 1] = 0.5, -50  # one expert takes more than its share, one nothing unless k asks for all
    for some in ("all", "most", "none"):
        valid = np.ones(T, np.uint8) if some == "all" else (np.arange(T) % 5 != 2).astype(np.uint8) if some == "most" else np.zeros(T, np.uint8)
        layer = gpu_layer(device, t)
        dv, db = torch.from_numpy(valid).cuda(), torch.from_numpy(bias).cuda()
        got = {}
        f32_joined = shared and kernel in ("mfma_f32", "generic")
        for way, call in (("inside", layer.forward_device), ("launch", layer.forward_device if f32_joined else layer.forward_timed)):
            if way == "launch" and f32_joined:   # (the timed forward's f32 shared expert, in launches of its own, has other tiles)
                layer.set_option(L.OPT_EXPLICIT_GATHER, 1)
            out = torch.full_like(x, 7.0)
            torch.cuda.synchronize()
            call(x.data_ptr(), T, out.data_ptr(), dv.data_ptr(), db.data_ptr())
            device.synchronize()
            got[way] = (out.cpu(), layer.cache(T, int(valid.sum())), layer.losses())
        assert layer.kernel_name() == kernel
        layer.set_option(L.OPT_EXPLICIT_GATHER, 0)
        if T <= 1000:   # (the call by itself: larger ones may have a launch, by the number of their tiles)
            assert (layer.forward_kernel_times(x.data_ptr(), T, out.data_ptr(), dv.data_ptr(), db.data_ptr())["dispatch"] == 0) == (E != 6)
        (out, cache, losses), (out2, cache2, losses2) = got["inside"], got["launch"]
        assert_routing_identical(cache, cache_as_ref(cache2))
        assert losses == losses2
        assert torch.equal(out.view(torch.int16 if act == "bf16" else torch.int32), out2.view(torch.int16 if act == "bf16" else torch.int32))
        if T <= 2049:
            assert_routing_identical(cache, oracle_layer(t).forward(t.x, valid=valid, router_bias=bias, threads=8))
        layer.close()


def cache_as_ref(cache):
    class Ref:
        pass
    r = Ref()
    for name in ("expert_of", "counts", "offsets", "perm_slot", "perm_token", "probabilities", "gate_of"):
        setattr(r, name, getattr(cache, name))
    r.lse = cache.log_sum_exp
    return r
