"""What the MoE layer is timed on: the calls a program makes through the public entry points.

Four kinds of call ("mode"):
  layer   MoELayer under torch.no_grad(): serving (decode and prefill) from fp32 masters.
  ops     ops.moe_forward on operands laid out once (packed bf16, or e4m3 with block scales), the
          way a server that loads ready weights calls it.
  step    a training step: MoELayer forward and backward after a weight update, so the step also
          rebuilds the kernels' operands from the fp32 masters.
  micro   a gradient-accumulation micro-step: forward and backward on unchanged weights.
Shapes are the configurations of the tests and the benchmark (32 experts top-4 SwiGLU; 64 skewed
experts; 128 sigmoid experts with a shared one; 128 fp8 experts) and the registered T3 expert
cells (256 ReLU^2 experts top-8 and a shared one, widths 1024 to 2048). Hidden states are N(0, 1)
in bf16, weights N(0, 0.02), as in the tests.
"""
import math

import torch

from nexttransformer_amd import _native as nat
from nexttransformer_amd import ops
from nexttransformer_amd.moe import MoELayer
from nexttransformer_amd.moe_recipe import MoERecipe

AUX_COEFF, Z_COEFF = 0.01, 0.001


def _shape(d, E, k, H, act, score="softmax", shared=0, zipf=0.0, dtype="bf16"):
    return dict(d=d, E=E, k=k, H=H, act=act, score=score, shared=shared, zipf=zipf, dtype=dtype)


SHAPES = {
    "e8": _shape(256, 8, 2, 512, "swiglu"),
    "e32": _shape(1024, 32, 4, 512, "swiglu"),
    "e64": _shape(2048, 64, 8, 1024, "swiglu", zipf=1.2),
    "e128": _shape(2048, 128, 8, 768, "swiglu", score="sigmoid", shared=1536),
    "e128-fp8": _shape(4096, 128, 8, 1536, "swiglu", dtype="fp8"),
    "e32-fp8": _shape(1024, 32, 4, 512, "swiglu", dtype="fp8"),
    "t3-L16": _shape(1024, 256, 8, 256, "relu2", shared=256),
    "t3-L20": _shape(1280, 256, 8, 320, "relu2", shared=320),
    "t3-L28": _shape(1792, 256, 8, 448, "relu2", shared=448),
    "t3-L32": _shape(2048, 256, 8, 512, "relu2", shared=512),
}


def listed():
    def case(name, mode, T, shape):
        return dict(name=name, mode=mode, T=T, **SHAPES[shape])

    return [
        # one token of one stream: latency and launches are all there is
        case("decode 1 of 32 experts", "layer", 1, "e32"),
        # a decode batch of 48 streams on the T3 cell: most experts touched, a row or two each
        case("decode 48 of 256 experts", "layer", 48, "t3-L20"),
        # an odd chunk of a prompt on the 128-expert layer with its shared expert
        case("chunk 777 of 128 experts", "ops", 777, "e128"),
        # 8 x 2048 tokens: the benchmark's forward
        case("prefill 16384 of 32 experts", "layer", 16384, "e32"),
        # the same batch through the T3 cell
        case("prefill 16384 of 256 experts", "layer", 16384, "t3-L20"),
        # the largest forward: 16 x 2048 tokens, the busiest expert at 8 times the mean
        case("skewed 32768 of 64 experts", "ops", 32768, "e64"),
        # fp8 serving: a decode batch (bound by the weights) and a prompt (bound by the products)
        case("fp8 decode 64 of 128 experts", "ops", 64, "e128-fp8"),
        case("fp8 prefill 4096 of 128 experts", "ops", 4096, "e128-fp8"),
        # a small model's training step, where the host and the launches weigh most
        case("step 512 of 8 experts", "step", 512, "e8"),
        # the training steps of the benchmark, each after a weight update
        case("step 16384 of 32 experts", "step", 16384, "e32"),
        case("step 16384 of 256 experts", "step", 16384, "t3-L20"),
        # a ragged micro-batch of gradient accumulation on a wider T3 cell
        case("micro 3001 of 256 experts", "micro", 3001, "t3-L28"),
    ]


def draw(rng):
    """One more case of the same ranges: the modes in use for each shape, token counts over their
    logarithm (most of them odd), never more work than the largest listed forward."""
    mode, shapes, low, high = rng.choice([
        ("layer", ("e8", "e32", "t3-L16", "t3-L20", "t3-L28"), 1, 16384),
        ("ops", ("e32", "e64", "e128", "t3-L16", "t3-L32"), 1, 16384),
        ("ops", ("e32-fp8", "e128-fp8"), 1, 4096),
        ("step", ("e8", "e32", "t3-L16", "t3-L20"), 64, 16384),
        ("micro", ("e8", "e32", "t3-L16", "t3-L28"), 64, 8192),
    ])
    T = round(math.exp(rng.uniform(math.log(low), math.log(high))))
    return dict(mode=mode, T=max(low, min(high, T)), **SHAPES[rng.choice(shapes)])


# -- inputs ------------------------------------------------------------------------------------

def _inputs(case, seed):
    """Hidden states, the output's gradient and fp32 weights, from the seed alone, on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    T, d, E, H, Hs = (case[n] for n in ("T", "d", "E", "H", "shared"))
    rows = 2 if case["act"] == "swiglu" else 1

    def normal(*shape, std=1.0, dtype=torch.float32):
        return torch.empty(shape, device="cuda", dtype=dtype).normal_(0.0, std, generator=g)

    v = dict(x=normal(T, d).to(torch.bfloat16), bias=None, shared_w1=None, shared_w2=None,
             router=normal(E, d, std=0.02), w1=normal(E, rows * H, d, std=0.02),
             w2=normal(E, d, H, std=0.02), grad=None)
    if Hs:
        v["shared_w1"] = normal(1, rows * Hs, d, std=0.02)
        v["shared_w2"] = normal(1, d, Hs, std=0.02)
    if case["zipf"]:
        v["bias"] = torch.tensor([-2.0 * case["zipf"] * math.log(r + 1) for r in range(E)],
                                 device="cuda", dtype=torch.float32)
    if case["mode"] in ("step", "micro"):
        v["grad"] = normal(T, d).to(torch.bfloat16)
    return v


def _layer(case, v):
    """An MoELayer with the case's weights as its fp32 masters."""
    layer = MoELayer(MoERecipe(
        layers=2, width=case["d"], heads=max(1, case["d"] // 64), sequence_len=max(2, case["T"]),
        global_batch_tokens=max(2, case["T"]), routed_experts=case["E"], top_k=case["k"],
        expert_width=case["H"], score_function=case["score"], activation=case["act"],
        shared_experts=1 if case["shared"] else 0, shared_expert_width=case["shared"] or None,
        expert_dtype=case["dtype"], allow_any_expert_width=True), 1)
    with torch.no_grad():
        layer.router.weight.copy_(v["router"])
        for i, e in enumerate(layer.experts.local_experts):
            e.linear_fc1.weight.copy_(v["w1"][i])
            e.linear_fc2.weight.copy_(v["w2"][i])
        if case["shared"]:
            layer.shared_experts.linear_fc1.weight.copy_(v["shared_w1"][0])
            layer.shared_experts.linear_fc2.weight.copy_(v["shared_w2"][0])
    layer.logit_bias = v["bias"]
    return layer


def _operands(case, v):
    """The weights as a server lays them out once for ops.moe_forward."""
    up = nat.EPI_SWIGLU if case["act"] == "swiglu" else nat.EPI_RELU2
    kw = dict(top_k=case["k"], activation=nat.ACT_SWIGLU if case["act"] == "swiglu" else nat.ACT_RELU2,
              score_fn=nat.SCORE_SIGMOID if case["score"] == "sigmoid" else nat.SCORE_SOFTMAX,
              aux_coeff=AUX_COEFF, z_coeff=Z_COEFF, logit_bias=v["bias"], packed=True)
    w = {}
    for name, epi in (("w1", up), ("w2", nat.EPI_NONE), ("shared_w1", up), ("shared_w2", nat.EPI_NONE)):
        if v[name] is None:
            continue
        if case["dtype"] == "fp8":
            q, scale = ops.quantize_fp8_blockwise(v[name])
            w[name], w[name + "_scale"] = ops.pack_expert_weights_fp8(q, epi), scale
        else:
            w[name] = ops.pack_expert_weights(v[name].to(torch.bfloat16), epi)
    kw.update((n, t) for n, t in w.items() if n not in ("w1", "w2"))
    return v["router"].t().contiguous(), w["w1"], w["w2"], kw


def prepare(case, seed):
    v = _inputs(case, seed)
    s = dict(mode=case["mode"], x=v["x"])
    if case["mode"] == "ops":
        s["router_t"], s["w1"], s["w2"], s["kw"] = _operands(case, v)
        return s
    s["layer"] = _layer(case, v)
    if case["mode"] == "layer":
        s["layer"].eval()
        with torch.no_grad():
            s["layer"].packed_weights()  # a server's weights do not change: laid out at load time
    else:
        s["x"].requires_grad_()
        s["grad"] = v["grad"]
        s["params"] = list(s["layer"].parameters())
        experts = s["layer"].experts.local_experts
        s["fc1"] = [e.linear_fc1.weight for e in experts]
        s["fc2"] = [e.linear_fc2.weight for e in experts]
    return s


# -- one pass ----------------------------------------------------------------------------------

def _whole(params):
    """The experts' gradients as one [E, rows, cols] tensor: without a copy where they are the
    consecutive slices of one stack, as the layer hands them out."""
    grads = [p.grad for p in params]
    a, z, n = grads[0], grads[-1], len(grads)
    if (a.is_contiguous() and a.untyped_storage().data_ptr() == z.untyped_storage().data_ptr()
            and z.storage_offset() - a.storage_offset() == (n - 1) * a.numel()):
        return a.as_strided((n,) + tuple(a.shape), (a.numel(),) + tuple(a.stride()),
                            a.storage_offset())
    return torch.stack(grads)


def run(s):
    if s["mode"] == "layer":
        with torch.no_grad():
            out, aux = s["layer"](s["x"])
        return dict(out=out, aux=aux, load=s["layer"].last_load)
    if s["mode"] == "ops":
        out, aux, state = ops.moe_forward(s["x"], s["router_t"], s["w1"], s["w2"], **s["kw"])
        return dict(out=out, aux=aux[0], load=state["counts"], ids=state["ids"],
                    weights=state["weights"])
    layer, x = s["layer"], s["x"]
    if s["mode"] == "step":  # the weights are new, as after an optimizer's in-place update
        torch.autograd.graph.increment_version(s["params"])
    for p in s["params"]:
        p.grad = None
    x.grad = None
    out, aux = layer(x)
    out.backward(s["grad"])
    r = dict(out=out.detach(), aux=aux, load=layer.last_load, dx=x.grad,
             router=layer.router.weight.grad, fc1=_whole(s["fc1"]), fc2=_whole(s["fc2"]))
    if layer.shared_experts is not None:
        r["shared_fc1"] = layer.shared_experts.linear_fc1.weight.grad
        r["shared_fc2"] = layer.shared_experts.linear_fc2.weight.grad
    return r


# -- what a pass cannot do without -------------------------------------------------------------

def work(case):
    T, d, E, k, H, Hs = (case[n] for n in ("T", "d", "E", "k", "H", "shared"))
    rows = 2 if case["act"] == "swiglu" else 1
    per_expert = (rows + 1) * H * d
    shared = (rows + 1) * Hs * d
    touched = E * (1.0 - (1.0 - k / E) ** T)  # experts that get a token, routing even
    flops = 2.0 * T * (k * per_expert + shared + E * d)
    if case["mode"] in ("layer", "ops"):
        size = 1 if case["dtype"] == "fp8" else 2
        bytes_ = touched * per_expert * size + shared * size + 4 * E * d + 4 * T * d
        if case["mode"] == "ops":
            bytes_ += 8 * T * k
        return dict(bytes=float(bytes_), flops=flops)
    weights = E * per_expert + shared + E * d
    read = 4 if case["mode"] == "step" else 2  # the fp32 masters, or their bf16 operands
    return dict(bytes=float((read + 4) * weights + 8 * T * d), flops=3.0 * flops)


def tolerance(case):
    """h, y and, in training, each gradient are rounded to bf16 on the way: measured against 64
    bits, forwards are up to 4.3e-3 off, fp8 ones and gradients up to 5.4e-3; about four times
    that. Routing is exact: loads and ids do not differ."""
    forward = case["mode"] in ("layer", "ops") and case["dtype"] == "bf16"
    return {"rel": 0.016 if forward else 0.02, "max": 0.25, "differ": 0.0}


# -- the same in 64 bits -----------------------------------------------------------------------

def _act(u, case):
    if case["act"] == "swiglu":
        gate, value = u.chunk(2, -1)
        return gate * torch.sigmoid(gate) * value
    return torch.relu(u).square()


def _e4m3(v, dims):
    """e4m3 values of v under one scale (largest magnitude / 448) over `dims`, dequantised."""
    v = v.float()
    top = v.abs().amax(dims, keepdim=True)
    scale = torch.where(top > 0, top / 448.0, torch.ones_like(top))
    return (v / scale).to(torch.float8_e4m3fn).double() * scale.double()


def _blocks(w):
    R, C = w.shape
    return _e4m3(w.view(R // 128, 128, C // 128, 128), (1, 3)).reshape(R, C)


def exact(case, seed):
    v = _inputs(case, seed)
    train = case["mode"] in ("step", "micro")
    fp8 = case["dtype"] == "fp8"
    T, d, E, k = (case[n] for n in ("T", "d", "E", "k"))
    names = ("router", "shared_w1", "shared_w2")
    x = v["x"].double()
    wr, s1, s2 = (None if v[n] is None else v[n].double() for n in names)
    w1 = [w.double() for w in v["w1"].unbind(0)] if train else v["w1"].unbind(0)
    w2 = [w.double() for w in v["w2"].unbind(0)] if train else v["w2"].unbind(0)
    if train:
        for t in [x, wr, s1, s2] + w1 + w2:
            if t is not None:
                t.requires_grad_()
    logits = x @ wr.t()
    if v["bias"] is not None:
        logits = logits + v["bias"].double()
    top, ids = logits.topk(k, -1)
    if case["score"] == "sigmoid":
        chosen, full = torch.sigmoid(top), torch.sigmoid(logits)
        weights, scores = chosen / chosen.sum(-1, keepdim=True), full / full.sum(-1, keepdim=True)
    else:
        weights, scores = top.softmax(-1), logits.softmax(-1)
    counts = torch.bincount(ids.reshape(-1), minlength=E)
    aux = (AUX_COEFF * E / (k * T * T) * (scores.sum(0) * counts.double()).sum()
           + Z_COEFF * torch.logsumexp(logits, -1).square().mean())

    def ffn(rows, a, b):
        if fp8:
            h = _act(rows @ _blocks(a).t(), case).to(torch.bfloat16)
            return _e4m3(h, -1) @ _blocks(b).t()
        return _act(rows @ a.double().t(), case) @ b.double().t()

    order = ids.reshape(-1).argsort(stable=True)  # expert by expert
    rows = _e4m3(x, -1) if fp8 else x
    xs = rows[order // k]
    parts, at = [], 0
    for e, n in enumerate(counts.tolist()):
        if n:
            parts.append(ffn(xs[at:at + n], w1[e], w2[e]))
            at += n
    y = torch.cat(parts)[order.argsort()].view(T, k, d)
    out = (y * weights[:, :, None]).sum(1)
    if s1 is not None:
        out = out + ffn(rows, s1[0], s2[0])
    if case["mode"] == "layer":
        return dict(out=out, aux=aux, load=None)
    if case["mode"] == "ops":
        return dict(out=out, aux=aux, load=None, ids=None, weights=weights)
    ((out * v["grad"].double()).sum() + aux).backward()
    zero = torch.zeros((), device=x.device, dtype=torch.float64)
    r = dict(out=out.detach(), aux=aux.detach(), load=None, dx=x.grad, router=wr.grad,
             fc1=torch.stack([w.grad if w.grad is not None else zero.expand_as(w) for w in w1]),
             fc2=torch.stack([w.grad if w.grad is not None else zero.expand_as(w) for w in w2]))
    if s1 is not None:
        r["shared_fc1"], r["shared_fc2"] = s1.grad[0], s2.grad[0]
    return r
