"""Timed workloads of the mixture-of-experts layer, through the public interface of ``rustingbrain_amd``.

The layer is used in four ways, and each has its cases:

* ``block``   — the feed-forward half of a transformer block on device rows (``MoeLayer.forward_block_device``):
  norm, layer and residual add, which is what a decode step or a prefill runs once per sparse layer;
* ``forward`` — the layer alone on device rows (``MoeLayer.forward_device``), optionally with a router bias that
  skews the load and a residual;
* ``host``    — ``MoeLayer.forward_train`` on host matrices, the reference's own signature, with the routing tables;
* ``train`` / ``train_host`` — one optimiser step's gradients: ``zero_grads``, then forward and backward for every
  micro-batch on device rows (block step) or host matrices (plain layer), then every weight gradient on the host,
  where the optimiser of a user of this package runs.

Layer sizes: the five benchmark workloads of ``rustingbrain_amd.synth.WORKLOADS`` and the default
``TransformerConfig`` (d_model 512, 8 experts top-2, expert width 352, shared expert, sequences of up to 2048 rows).
"""
from __future__ import annotations

import math

import torch

import rustingbrain_amd as rb
from rustingbrain_amd import _lib as L

_device = None


def _dev():
    """One handle for the GPU, as a program with many layers keeps: every layer's work goes to its one stream."""
    global _device
    if _device is None:
        _device = rb.Device.open(0)
    return _device


def _case(kind, d, experts, top_k, d_ff, shared, tokens, rows, weights, **more):
    c = {"kind": kind, "d": d, "experts": experts, "top_k": top_k, "d_ff": d_ff, "shared": shared, "tokens": tokens,
         "rows": rows, "weights": weights, "quantized_router": False, "padding": 0.0, "skew": 0.0, "micro": 1}
    c.update(more)
    return c


def listed():
    return [
        # one token of one conversation, default model: the smallest call there is, all latency
        _case("block", 512, 8, 2, 352, 352, 1, "bf16", "bf16", name="decode_one_row"),
        # a batch of eight decode steps (the benchmark's decode workload)
        _case("forward", 768, 8, 2, 1408, 1408, 8, "bf16", "bf16", name="decode_batch"),
        # a full decode batch of a model quantized in memory: int8 experts and int8 router
        _case("block", 768, 8, 2, 1408, 0, 32, "bf16", "int8", quantized_router=True, name="decode_quantized"),
        # a serving step that mixes decode rows with short prompts, padded to the batch: a few hundred ragged rows
        _case("block", 768, 16, 2, 1408, 0, 203, "bf16", "bf16", padding=0.1, name="serving_mixed"),
        # the README's layer in the reference's own precision
        _case("forward", 512, 8, 2, 1408, 0, 1024, "f32", "f32", name="f32_forward"),
        # the prompt of one full sequence through the default model
        _case("block", 512, 8, 2, 352, 352, 2048, "bf16", "bf16", name="default_prefill"),
        # int8 checkpoint, bf16 rows, a medium batch
        _case("forward", 768, 8, 2, 1408, 0, 4096, "bf16", "int8", name="int8_forward"),
        # the headline: a large prefill with one expert taking 30 % of the assignments
        _case("forward", 768, 16, 2, 1408, 0, 8192, "bf16", "bf16", skew=0.3, name="prefill_skewed"),
        # many narrow experts, six a token, and a shared expert: the largest forward
        _case("forward", 1024, 64, 6, 704, 1408, 16384, "bf16", "bf16", name="fine_grained"),
        # the reference's call: f32 host matrix in (three padded sequences), f32 matrix and routing tables out
        _case("host", 768, 8, 2, 1408, 0, 1533, "f32", "int8", padding=0.1, name="host_forward"),
        # gradients of one step on host matrices in f32, the reference's own way to train
        _case("train_host", 512, 8, 2, 1408, 0, 1024, "f32", "f32", name="host_training"),
        # gradients of one step in bf16: four micro-batches of 8192 rows accumulated on the device
        _case("train", 768, 16, 2, 1408, 0, 8192, "bf16", "bf16", micro=4, name="training"),
    ]


# layer shapes: (d_model, experts, top_k, d_ff, shared width)
_SHAPES = [(512, 8, 2, 352, 352), (512, 8, 2, 1408, 0), (768, 8, 2, 1408, 1408), (768, 16, 2, 1408, 0),
           (1024, 64, 6, 704, 1408)]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        if rng.random() < 0.6:
            d, e, k, f, fs = rng.choice(_SHAPES)
        else:
            d = rng.choice([256, 512, 768, 1024])
            e = rng.choice([4, 8, 16, 32])
            k = rng.choice([1, 2, 4])
            # two thirds rounded the way transformer configurations round, the rest the unrounded 8/3 of a width
            f = rng.choice([256, 352, 704, 1408]) if rng.random() < 0.67 else 8 * d // rng.choice([3, 6, 9])
            fs = rng.choice([0, 0, f])
        kind = rng.choice(["block", "block", "forward", "forward", "forward", "host", "train", "train_host"])
        rows, weights = rng.choice([("bf16", "bf16"), ("bf16", "bf16"), ("bf16", "int8"), ("f32", "bf16"),
                                    ("f32", "int8"), ("f32", "f32")])
        if kind == "train":
            t = _log_int(rng, 512, 8192)
            rows, weights = rng.choice([("bf16", "bf16"), ("bf16", "bf16"), ("f32", "f32")])
        elif kind == "train_host":
            t = _log_int(rng, 128, 4096)
            rows, weights = rng.choice([("f32", "f32"), ("f32", "f32"), ("f32", "bf16")])
        elif kind == "host":
            t = _log_int(rng, 1, 8192)
        else:
            t = _log_int(rng, 1, 16384)
        # (with one expert per token the router's gradient is zero on paper and rounding noise in f32)
        if kind.startswith("train") and (e > 16 or k == 1):
            continue
        c = _case(kind, d, e, k, f, fs, t, rows, weights,
                  quantized_router=weights == "int8" and rng.random() < 0.5,
                  padding=rng.choice([0.0, 0.0, 0.1, 0.3]) if t > 8 and kind != "train" else 0.0,
                  skew=0.3 if kind == "forward" and t >= 256 and 0.3 * k < 0.9 and rng.random() < 0.3 else 0.0,
                  micro=rng.choice([1, 2]) if kind == "train" else 1)
        # no dearer than the largest listed case (f32 products run at a sixteenth of the bf16 rate)
        if work(c)["flops"] * (8 if rows == "f32" and weights == "f32" else 1) <= 9e11 and work(c)["bytes"] <= 1.2e9:
            return c


# ----------------------------------------------------------------------------- inputs
def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std


def _xavier(g, rows, cols):
    a = math.sqrt(6.0 / (rows + cols))
    return (torch.rand((rows, cols), generator=g, device="cuda", dtype=torch.float32) * 2 - 1) * a


def _quantize(w):
    """One symmetric int8 row per output channel, scale absmax / 127 (what an int8 checkpoint holds)."""
    s = w.abs().amax(dim=1) / 127.0
    q = torch.clamp(torch.round(w / s[:, None]), -127, 127).to(torch.int8)
    return q.cpu().numpy(), s.cpu().numpy()


def _load_expert(c, g, width, put, put_q8):
    d = c["d"]
    mats = [_xavier(g, width, d), _xavier(g, width, d), _xavier(g, d, width)]
    if c["weights"] == "int8":
        put_q8(*[a for m in mats for a in _quantize(m)])
    else:
        put(*[m.cpu().numpy() for m in mats])


def _rows_of(c, t):
    return t.to(torch.bfloat16) if c["rows"] == "bf16" else t


def _bias_for(c, x, router):
    """A bias on expert 0's logit that gives it the share ``skew`` of all assignments."""
    logits = x.float() @ router.T
    others = logits[:, 1:].topk(c["top_k"], dim=1).values[:, -1]
    need = (others - logits[:, 0]).sort().values
    b = torch.zeros(c["experts"], device="cuda", dtype=torch.float32)
    b[0] = need[min(len(need) - 1, int(c["skew"] * c["top_k"] * len(need)))] + 1e-4
    return b


class _State:
    pass


def prepare(case, seed):
    c = case
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    d, e, t = c["d"], c["experts"], c["tokens"]
    training = c["kind"].startswith("train")
    s = _State()
    s.case = c
    config = rb.MoeConfig.new(e, c["top_k"], c["d_ff"]).with_shared_expert(c["shared"] > 0)
    # a serving layer takes prompts of up to 2048 rows besides its decode steps
    s.layer = rb.MoeLayer(d, config, _dev(), act_dtype=c["rows"], weight_dtype=c["weights"],
                          max_tokens=t if training else max(t, 2048), shared_d_ff=c["shared"])
    if training:
        s.layer.enable_training()
    router = _normal(g, (e, d), 0.02)
    if c["weights"] != "f32":
        router = router.to(torch.bfloat16).float()
    if c["quantized_router"]:
        s.layer.set_router_q8(*_quantize(router))
    else:
        s.layer.set_router(router.cpu().numpy())
    for i in range(e):
        _load_expert(c, g, c["d_ff"], lambda *m: s.layer.set_expert(i, *m), lambda *m: s.layer.set_expert_q8(i, *m))
    if c["shared"]:
        _load_expert(c, g, c["shared"], s.layer.set_shared, s.layer.set_shared_q8)
    if c["kind"] in ("block", "train"):
        s.layer.set_feed_forward_norm((1.0 + _normal(g, (d,), 0.1)).cpu().numpy(), 1e-6)
    s.x = [_rows_of(c, _normal(g, (t, d))) for _ in range(c["micro"])]
    s.valid = None
    if c["padding"] > 0:
        s.valid = torch.ones(t, dtype=torch.bool, device="cuda")
        s.valid[torch.randperm(t, generator=g, device="cuda")[:round(c["padding"] * t)]] = False
    s.bias = _bias_for(c, s.x[0], router) if c["skew"] > 0 else None
    s.grad = [_rows_of(c, _normal(g, (t, d))) for _ in range(c["micro"])] if training else []
    if c["kind"] in ("host", "train_host"):
        s.x = [v.float().cpu().numpy() for v in s.x]
        s.grad = [v.float().cpu().numpy() for v in s.grad]
        s.layout = rb.Layout(valid=None if s.valid is None else s.valid.cpu().numpy())
    else:
        s.out = [torch.empty_like(v) for v in s.x]
        s.grad_in = [torch.empty_like(v) for v in s.grad]
        s.valid = None if s.valid is None else s.valid.to(torch.uint8)
    torch.cuda.synchronize()
    return s


# ----------------------------------------------------------------------------- one pass
def _ptr(t):
    return 0 if t is None else t.data_ptr()


def _weight_grads(layer, shared, norm):
    g = {"router": layer.weight_grad(L.W_ROUTER)}
    for name, which in (("gate", L.W_GATE), ("up", L.W_UP), ("down", L.W_DOWN)):
        g[name] = [layer.weight_grad(which, i) for i in range(layer.config.num_experts)]
    if shared:
        g["shared"] = [layer.weight_grad(w) for w in (L.W_SHARED_GATE, L.W_SHARED_UP, L.W_SHARED_DOWN)]
    if norm:
        g["norm"] = layer.weight_grad(L.W_NORM)
    return g


def run(state):
    c, layer, t = state.case, state.layer, state.case["tokens"]
    kind = c["kind"]
    if kind == "block":
        layer.forward_block_device(state.x[0].data_ptr(), t, state.out[0].data_ptr(), _ptr(state.valid))
        return state.out[0]
    if kind == "forward":
        layer.forward_device(state.x[0].data_ptr(), t, state.out[0].data_ptr(), _ptr(state.valid), _ptr(state.bias))
        return state.out[0]
    if kind == "host":
        out, cache = layer.forward_train(state.x[0], state.layout)
        return {"out": out, "expert_of": cache.expert_of, "gate_of": cache.gate_of, "counts": cache.counts,
                "perm_token": cache.perm_token, "probabilities": cache.probabilities,
                "log_sum_exp": cache.log_sum_exp, "loss": cache.auxiliary_loss()}
    layer.zero_grads()
    if kind == "train_host":
        out, cache = layer.forward_train(state.x[0], state.layout)
        grad_in = layer.backward(state.grad[0])
        return {"out": out, "loss": cache.auxiliary_loss(), "grad_input": grad_in,
                "grads": _weight_grads(layer, c["shared"] > 0, False)}
    for x, out, grad, grad_in in zip(state.x, state.out, state.grad, state.grad_in):
        layer.forward_block_device(x.data_ptr(), t, out.data_ptr())
        layer.backward_block_device(grad.data_ptr(), t, grad_in.data_ptr())
    return {"out": state.out, "grad_input": state.grad_in, "grads": _weight_grads(layer, c["shared"] > 0, True)}


# ----------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    c = case
    d, e, k, f, fs, t = c["d"], c["experts"], c["top_k"], c["d_ff"], c["shared"], c["tokens"]
    training = c["kind"].startswith("train")
    size = {"f32": 4, "bf16": 2, "int8": 1}
    # experts that take rows: all of them for large batches, the expected number for a few tokens
    touched = e * (1.0 - (1.0 - k / e) ** t)
    weights = 3.0 * d * (touched * f + fs)
    rows = float(t) * d * size[c["rows"]]
    bytes_ = weights * size[c["weights"]] + e * d * 4.0 + 2.0 * c["micro"] * rows
    routed = t * k * (1.0 - c["padding"])
    flops = c["micro"] * (6.0 * d * (routed * f + t * fs) + 2.0 * t * e * d)
    if c["kind"] == "host":
        bytes_ += t * (e + 1.0 + 3.0 * k) * 4.0
    if training:
        flops *= 3.0
        bytes_ += 2.0 * c["micro"] * rows + (3.0 * d * (e * f + fs) + e * d) * 4.0
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    # Expert products in bf16 (f32 accumulation, bf16 hidden and output rows): 2^-9 a rounding, a few in a row.
    # All-f32 layers: sums of a few thousand f32 terms in another order.  Routing tables are whole numbers: the same.
    return {"rel": 1e-5} if case["rows"] == "f32" and case["weights"] == "f32" else {"rel": 1e-2}
