"""What programs built on this library spend their time on, as cases to be timed: the quantised linear layers of a
decoder in inference and in fine-tuning, and the optimizer's step on their latent weights.

A case names a kind of work and its sizes. ``prepare`` builds the layers and inputs a program has in hand, ``run`` takes
one pass through the public entry points (the modules of ``latentq_llm_amd.quant``, ``QuantLlamaMLP``, ``MyAdam``).

kind        one pass
decode      the seven linear layers of ``layers`` decoder layers (int4 weights, gated MLP) on 1 to 16 tokens, one
            from every sequence of a batch: what a generation loop does for each new token
prefill     the same seven layers of one decoder layer on a prompt, 17 to 8192 tokens in all
infer8      the six linear layers of one decoder layer with int8 weights and activations (plain MLP, biases) in
            inference, one token to a prompt
train_mlp   a gated MLP block with int4 weights in fine-tuning: two micro-batches forward and backward, the second
            accumulated onto the weight gradients of the first
train_linear  the same for one linear layer: int4 weights, int8 weights and activations, or quantisation-aware
optim       one optimizer step on the six weights of such a decoder layer: 8-bit moments, and the latent weight as
            int4 codes with stochastic rounding, int4 codes + 4-bit residual, int8 codes + 4-bit residual, or bf16

Attention, norms and residual additions are the program's own and left out: a layer's output goes straight to the next.
Weights, scales and zero points are drawn as the repository's benchmark draws them, activations are N(0, 1).
"""
import torch

from latentq_llm_amd.fused_mlp import QuantLlamaMLP
from latentq_llm_amd.quant import GradientQTensor, MyAdam, QLinearA8W8, QLinearA16W4, QLinearQAT

BF16 = torch.bfloat16
MICRO_BATCHES = 2


def listed():
    return [
        # a chat with one user: one token at a time through layers of 4096 / 11008
        {"name": "decode_1", "kind": "decode", "tokens": 1, "layers": 2, "hidden": 4096, "inter": 11008},
        # a dozen sequences generated together
        {"name": "decode_12", "kind": "decode", "tokens": 12, "layers": 2, "hidden": 4096, "inter": 11008},
        # a short question
        {"name": "prefill_45", "kind": "prefill", "tokens": 45, "hidden": 4096, "inter": 11008},
        # a page of text, a length nobody chose
        {"name": "prefill_1019", "kind": "prefill", "tokens": 1019, "hidden": 4096, "inter": 11008},
        # a batch of long prompts: the largest
        {"name": "prefill_8192", "kind": "prefill", "tokens": 8192, "hidden": 4096, "inter": 11008},
        # fine-tuning at the benchmark's size: 4 x 512 tokens, gradients kept in bf16
        {"name": "train_mlp_2048", "kind": "train_mlp", "tokens": 2048, "hidden": 4096, "inter": 11008, "gbit": 16},
        # fine-tuning on unpadded examples of a smaller model, gradients kept in int8
        {"name": "train_mlp_500", "kind": "train_mlp", "tokens": 500, "hidden": 2048, "inter": 5504, "gbit": 8},
        # the benchmark's smallest layer in training
        {"name": "train_w4_small", "kind": "train_linear", "schema": "a16w4", "tokens": 1024, "n": 3072, "k": 768, "bias": True, "gbit": 16,
         "act": "per_tensor"},
        # the benchmark's 8-bit layer in training
        {"name": "train_w8", "kind": "train_linear", "schema": "a8w8", "tokens": 2048, "n": 8192, "k": 2048, "bias": True, "gbit": 16,
         "act": "per_tensor"},
        # four sequences generated together on 8-bit layers
        {"name": "infer8_4", "kind": "infer8", "tokens": 4, "hidden": 2048, "act": "per_tensor"},
        # the two 4-bit optimizer modes at the size of the benchmark's requantizer and optimizer legs
        {"name": "optim_sr", "kind": "optim", "latent": "sr", "hidden": 2048},
        {"name": "optim_w4", "kind": "optim", "latent": "w4", "hidden": 2048},
    ]


def _log(rng, lo, hi):
    """An integer of lo..hi, spread over its logarithm."""
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(("decode", "prefill", "infer8", "train_mlp", "train_linear", "optim"))
    hidden = 256 * rng.randint(4, 16)
    inter = min(11008, 128 * rng.randint(2 * hidden // 128, 4 * hidden // 128))  # any multiple of the 128-element group
    act = rng.choice(("per_tensor", "per_tensor", "per_token"))
    if kind == "decode":
        return {"kind": kind, "tokens": rng.randint(1, 16), "layers": rng.randint(1, 3), "hidden": hidden, "inter": inter}
    if kind == "prefill":
        return {"kind": kind, "tokens": _log(rng, 17, 8192), "hidden": hidden, "inter": inter}
    if kind == "infer8":
        return {"kind": kind, "tokens": _log(rng, 1, 2048), "hidden": 256 * rng.randint(3, 10), "act": act}
    if kind == "train_mlp":
        # padded batches (a multiple of 64 tokens) as often as unpadded ones
        tokens = 64 * _log(rng, 1, 32) if rng.random() < 0.5 else _log(rng, 64, 2048)
        return {"kind": kind, "tokens": tokens, "hidden": hidden, "inter": inter, "gbit": rng.choice((16, 8))}
    if kind == "train_linear":
        tokens = 64 * _log(rng, 1, 64) if rng.random() < 0.5 else _log(rng, 64, 4096)
        n, k = rng.choice(((hidden, hidden), (inter, hidden), (hidden, inter)))
        schema = rng.choice(("a16w4", "a8w8", "qat"))
        return {"kind": kind, "schema": schema, "tokens": tokens, "n": n, "k": k, "bias": rng.random() < 0.5,
                "gbit": 16 if schema == "qat" else rng.choice((16, 8)), "act": act if schema == "a8w8" else "per_tensor"}
    return {"kind": kind, "latent": rng.choice(("sr", "w4", "w8", "bf16")), "hidden": 256 * rng.randint(3, 10)}


# ------------------------------------------------------------------------------------------- layers and inputs --
class _Draws:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, shape, std=1.0):
        return torch.empty(shape, dtype=BF16, device="cuda").normal_(0, std, generator=self.gen)

    def integers(self, lo, hi, shape, dtype):
        return torch.randint(lo, hi, shape, generator=self.gen, device="cuda", dtype=dtype)


def _set_bias(layer, d):
    if layer.bias is not None:
        layer.bias.data = d.normal((layer.output_features,), 0.1)


def _w4(n, k, d, bias=False, lbit=4, gbit=16):
    layer = QLinearA16W4(k, n, bias=bias, lbit=lbit, gbit=gbit)
    groups = n * k // 128
    layer.scales.data = d.normal((groups, 1), 0.02).abs_().div_(7).clamp_(min=2.0 ** -12)
    layer.zeros.data = d.integers(6, 10, (groups, 1), torch.int32).to(BF16)
    layer.weight.set_value(d.integers(-128, 128, (n * k // 2,), torch.int8), [layer.scales, layer.zeros, layer.wshape])
    _set_bias(layer, d)
    return layer


def _w8(n, k, d, bias=True, lbit=4, gbit=16, act="per_tensor"):
    layer = QLinearA8W8(k, n, bias=bias, lbit=lbit, gbit=gbit)
    layer.act_quant = act
    layer.qscales.data = d.normal((n, 1), 3e-4).abs_().clamp_(min=1e-5)
    layer.weight.set_value(d.integers(-127, 128, (n, k), torch.int8), layer.qscales)
    _set_bias(layer, d)
    return layer


def _qat(n, k, d, bias=True):
    layer = QLinearQAT(k, n, bias=bias)
    layer.qscales.data = d.normal((n, 1), 3e-4).abs_().clamp_(min=1e-5)
    layer.weight.data = (d.normal((n, k), 40.0) * layer.qscales).to(BF16)
    _set_bias(layer, d)
    return layer


def _mlp(hidden, inter, d, gbit=16):
    return QuantLlamaMLP(_w4(inter, hidden, d, gbit=gbit), _w4(hidden, inter, d, gbit=gbit), _w4(inter, hidden, d, gbit=gbit))


def _gated_layer(hidden, inter, d):
    return [_w4(hidden, hidden, d) for _ in range(4)] + [_mlp(hidden, inter, d)]


def _plain_shapes(hidden):
    """(out, in) of a plain decoder layer's six linear layers."""
    return [(hidden, hidden)] * 4 + [(4 * hidden, hidden), (hidden, 4 * hidden)]


# --------------------------------------------------------------------------------------------------- prepare / run --
def prepare(case, seed):
    d = _Draws(seed)
    kind = case["kind"]
    state = {"kind": kind, "seed": seed}
    if kind in ("decode", "prefill"):
        state["layers"] = [_gated_layer(case["hidden"], case["inter"], d) for _ in range(case.get("layers", 1))]
        shape = (case["tokens"], 1) if kind == "decode" else (1, case["tokens"])
        state["x"] = d.normal(shape + (case["hidden"],))
    elif kind == "infer8":
        state["layers"] = [_w8(n, k, d, act=case["act"]) for n, k in _plain_shapes(case["hidden"])]
        state["x"] = d.normal((1, case["tokens"], case["hidden"]))
    elif kind in ("train_mlp", "train_linear"):
        if kind == "train_mlp":
            block = _mlp(case["hidden"], case["inter"], d, case["gbit"])
            trained, n, k = [block.gate_proj, block.up_proj, block.down_proj], case["hidden"], case["hidden"]
        else:
            n, k = case["n"], case["k"]
            if case["schema"] == "a16w4":
                block = _w4(n, k, d, case["bias"], gbit=case["gbit"])
            elif case["schema"] == "a8w8":
                block = _w8(n, k, d, case["bias"], gbit=case["gbit"], act=case["act"])
            else:
                block = _qat(n, k, d, case["bias"])
            trained = [block]
        for layer in trained:
            layer.add_hook()
        state.update(block=block, trained=trained)
        state["batches"] = [(d.normal((1, case["tokens"], k)), d.normal((1, case["tokens"], n), 1e-3)) for _ in range(MICRO_BATCHES)]
    else:
        weights = []
        for n, k in _plain_shapes(case["hidden"]):
            if case["latent"] == "bf16":
                w = _qat(n, k, d, bias=False).weight
            elif case["latent"] == "w8":
                w = _w8(n, k, d, bias=False).weight
            else:
                w = _w4(n, k, d, lbit=0 if case["latent"] == "sr" else 4).weight
            weights.append(w)
        state["weights"] = weights
        state["grads"] = [d.normal(tuple(w.shape), 1e-3) for w in weights]
        state["opt"] = MyAdam([{"params": weights}], lr=1e-5, betas=(0.9, 0.95), obit=8, sr_seed=seed)
        for _ in range(2):  # training is under way: moments and residuals hold values
            _step(state)
    return state


def _step(state):
    for w, g in zip(state["weights"], state["grads"]):
        w.grad = g
    state["opt"].step()


def _run_inference(state):
    out, x = [], state["x"]
    with torch.no_grad():
        for layer in state["layers"]:
            if state["kind"] == "infer8":
                out.append(layer(x))
                x = out[-1] if len(out) > 3 else x  # q, k, v read the same input
            else:
                q, k, v, o, mlp = layer
                out += [q(x), k(x), v(x)]
                x = mlp(o(out[-1]))
                out.append(x)
    return out


def _run_training(state):
    # the window starts without gradients; its rounding noise (int8 gradients) is seeded, as torch.manual_seed would
    GradientQTensor.noise_seed, GradientQTensor._noise_offset = state["seed"], 0
    for layer in state["trained"]:
        if isinstance(layer.weight.grad, GradientQTensor):
            layer.weight.grad.zero()
        else:
            layer.weight.grad = None
    out = []
    for x, dy in state["batches"]:
        x = x.detach().requires_grad_(True)
        y = state["block"](x)
        y.backward(dy)
        out += [y.detach(), x.grad]
    for layer in state["trained"]:
        g = layer.weight.grad
        out += [g.qdata, g.scale] if isinstance(g, GradientQTensor) else [g]
    return out


def _run_optimizer(state):
    _step(state)
    out = []
    for w in state["weights"]:
        s = state["opt"].state[w]
        out += [w.data, s["state1"], s["qmap1"], s["absmax1"], s["state2"], s["qmap2"], s["absmax2"]]
        residual = getattr(w, "residual", None)
        if residual is not None:
            out.append(residual.residual_int)
    return out


def run(state):
    if state["kind"] == "optim":
        return _run_optimizer(state)
    return _run_training(state) if state["kind"].startswith("train") else _run_inference(state)


# ------------------------------------------------------------------------------------------------------ accounting --
def _weight_bytes(n, k, schema):
    return n * k / 2 + 4 * n * k / 128 if schema == "a16w4" else n * k + 2 * n if schema == "a8w8" else 2 * n * k + 2 * n


def work(case):
    kind = case["kind"]
    if kind == "optim":
        # gradient read; two uint8 moments and the latent weight (codes, residual) read and written, per element; group scales
        n = sum(a * b for a, b in _plain_shapes(case["hidden"]))
        per = {"sr": 2 + 4 + 1, "w4": 2 + 4 + 1 + 1, "w8": 2 + 4 + 2 + 1, "bf16": 2 + 4 + 4}[case["latent"]]
        scales = 4 / 128 if case["latent"] in ("sr", "w4") else 0
        return {"bytes": n * (per + scales + 32 / 2048), "flops": 0}
    m = case["tokens"]
    if kind == "train_linear":
        shapes, schema = [(case["n"], case["k"])], case["schema"]
        io = case["n"] + case["k"]
    elif kind == "infer8":
        shapes, schema = _plain_shapes(case["hidden"]), "a8w8"
        io = 7 * case["hidden"]  # the input, q, k, v, o, the up and the down projection's results, less what stays inside
    else:
        h, i = case["hidden"], case["inter"]
        shapes, schema = [(i, h), (i, h), (h, i)], "a16w4"
        io = 2 * h
        if kind in ("decode", "prefill"):
            shapes, io = shapes + [(h, h)] * 4, 5 * h
    params = sum(n * k for n, k in shapes)
    weights = sum(_weight_bytes(n, k, schema) for n, k in shapes)
    if kind.startswith("train"):
        # y, dx and dW of every micro-batch; x, dy read, y, dx written; the weights and their gradient once
        return {"bytes": weights + params * (case["gbit"] / 8) + MICRO_BATCHES * 4 * m * io, "flops": MICRO_BATCHES * 6 * m * params}
    layers = case.get("layers", 1)
    return {"bytes": layers * (weights + 2 * m * io), "flops": layers * 2 * m * params}


def tolerance(case):
    """Optimizer state is bytes and their block parameters, bit for bit. Elsewhere bf16 results of sums taken in another
    order, rounded at other points of a chain of layers. Measured against the same path in 64 bits: 2e-3 for one layer,
    4e-3 for a block in prefill or training, 1e-2 after two layers in decoding; where activations are rounded to int8 a tie
    that falls the other way moves a value by a whole code (6e-3 to 8e-3 for a layer, more down a chain). int8 gradients
    may round to the neighbouring code."""
    if case["kind"] == "optim":
        return "exact"
    if case["kind"] == "infer8" or case.get("schema") in ("a8w8", "qat"):
        return {"rel": 2.5e-2, "max": 0.4, "differ": 5e-3}
    if case["kind"] == "decode":
        return {"rel": 2e-2, "max": 0.16}
    return {"rel": 1.5e-2, "max": 0.12, "differ": 5e-3}
