"""What the quantized linears of this framework are used for, as cases that can be timed and compared.

Every case is one pass of a user's program through the public entry points: a layer in inference, a layer's training
step, the two layers whose producer (RMSNorm, SwiGLU) is fused into them, a quantizer module on its own, and the Llama
model in evaluation.  Widths are those of the repository's model configurations (640, 1536, 1728, 4096, 4608, 8192,
11008, ...) and of their neighbourhood; token counts run from one decoded batch to a large training micro-batch.

A whole training step of the model is not a case of its own: behind the first few layers two correct implementations
round different FP4 codes, so the gradients of the early layers are not comparable.  Its layers are all here instead, in
each role that they have in the model."""
import math
import random

import torch

import quartet_amd as q
from quartet_amd.fused import rmsnorm_linear, swiglu_linear
from quartet_amd.llama import Llama, RMSNorm, llama_30m

PRODUCTION_SCHEME = "Q(E)Q(Wt)t_Q(Et)Q(Xt)t"
ERROR_ONLY_SCHEME = "Q(E)W_Q(Et)X"
LARGEST = 8192 * 4096 * 11008  # tokens * in * out of the largest listed layer


def listed():
    return [
        # one decoding step of a batch of eight sequences: the weight is constant and stays packed
        {"name": "decode 8x4096x4096", "kind": "infer", "tokens": 8, "in": 4096, "out": 4096, "hd": 32},
        # a prompt being processed: token counts are whatever the prompts add up to
        {"name": "prefill 1000x1536x8192", "kind": "infer", "tokens": 1000, "in": 1536, "out": 8192, "hd": 32},
        # training step on one short sequence of the small model (fp32 master weights, bf16 autocast): host and launches count
        {"name": "train 512x640x1920", "kind": "train", "tokens": 512, "in": 640, "out": 1920, "hd": 32, "amp": True},
        # training step of a 7B-class attention projection: the repository's benchmark workload
        {"name": "train 8192x4096x4096", "kind": "train", "tokens": 8192, "in": 4096, "out": 4096, "hd": 32, "amp": False},
        # training step of a 7B-class MLP projection
        {"name": "train 8192x4096x11008", "kind": "train", "tokens": 8192, "in": 4096, "out": 11008, "hd": 32, "amp": False},
        # the small model's MLP projection (hidden width 1728) on packed sequences that do not fill whole tiles
        {"name": "train 16480x1728x640", "kind": "train", "tokens": 16480, "in": 1728, "out": 640, "hd": 32, "amp": True},
        # Hadamard blocks of 128, the widest rotation the quantizers offer
        {"name": "train hd128 8192x1536x4608", "kind": "train", "tokens": 8192, "in": 1536, "out": 4608, "hd": 128, "amp": True},
        # the scheme that quantizes only the error signal in backward
        {"name": "error-only 4096x4096x4096", "kind": "error_only", "tokens": 4096, "in": 4096, "out": 4096, "hd": 32, "amp": False},
        # RMSNorm with the residual sum in front of it, into the attention's input projection of the 800 M model
        {"name": "norm+linear 16384x1536x4608", "kind": "norm_linear", "tokens": 16384, "in": 1536, "out": 4608, "hd": 32, "amp": True},
        # SwiGLU into the MLP's output projection of the 800 M model
        {"name": "swiglu+linear 16384x4096x1536", "kind": "swiglu_linear", "tokens": 16384, "in": 4096, "out": 1536, "hd": 32, "amp": True},
        # a quantizer module by itself (pseudo-quantization and its straight-through backward), as quantization studies use it
        {"name": "quantizer hd64 16384x4096", "kind": "quantizer", "which": "quest", "tokens": 16384, "in": 4096, "hd": 64},
        # evaluation of the 30 M model: forward pass, logits and loss
        {"name": "llama30m eval 8x512", "kind": "llama_eval", "batch": 8, "seq": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: mostly multiples of 128, every third an odd or even multiple of 64 (as the hidden width 1728)."""
    unit = 128 if rng.random() < 2 / 3 else 64
    return max(lo, _log_int(rng, lo, hi) // unit * unit)


def _tokens(rng, lo, hi, unit):
    """Tokens of a training step: whole sequences mostly, every third packed to a multiple of `unit` only."""
    t = _log_int(rng, lo, hi)
    unit = max(unit, 256) if rng.random() < 2 / 3 else unit
    return max(lo, t // unit * unit)


def draw(rng):
    kind = rng.choice(["infer", "infer", "train", "train", "train", "train_hd", "error_only", "norm_linear", "swiglu_linear",
                       "quantizer", "llama_eval"])
    if kind == "llama_eval":
        return {"kind": kind, "batch": _log_int(rng, 1, 8), "seq": _log_int(rng, 64, 512)}
    while True:
        if kind == "infer":
            case = {"kind": kind, "tokens": _log_int(rng, 1, 8192), "in": _width(rng, 512, 11008), "out": _width(rng, 512, 11008), "hd": 32}
        elif kind == "quantizer":
            hd = rng.choice([32, 64, 128])
            case = {"kind": kind, "which": rng.choice(["quest", "quest", "albert"]), "tokens": _log_int(rng, 256, 32768),
                    "in": _log_int(rng, 512, 8192) // hd * hd, "hd": hd}
        elif kind == "train_hd":
            hd = rng.choice([64, 128])
            case = {"kind": "train", "tokens": _tokens(rng, 512, 16384, hd), "in": _width(rng, 512, 8192) // hd * hd,
                    "out": _width(rng, 512, 8192) // hd * hd, "hd": hd, "amp": rng.random() < 0.5}
        elif kind == "error_only":
            case = {"kind": kind, "tokens": _tokens(rng, 512, 16384, 64), "in": _width(rng, 512, 8192), "out": _width(rng, 512, 8192),
                    "hd": 32, "amp": rng.random() < 0.5}
        elif kind in ("norm_linear", "swiglu_linear"):
            case = {"kind": kind, "tokens": _tokens(rng, 512, 32768, 32), "in": _width(rng, 512, 4096), "out": _width(rng, 512, 8192),
                    "hd": 32, "amp": True}
        else:
            case = {"kind": "train", "tokens": _tokens(rng, 256, 32768, 32), "in": _width(rng, 512, 11008), "out": _width(rng, 512, 11008),
                    "hd": 32, "amp": rng.random() < 0.5}
        if case["tokens"] * case["in"] * case.get("out", 1) <= LARGEST * (0.25 if kind == "error_only" else 1.0):
            return case


def _normal(gen, *shape, scale=1.0, dtype=torch.bfloat16):
    return (torch.randn(*shape, generator=gen, device="cuda") * scale).to(dtype)


def _activations(gen, rows, cols, dtype=torch.bfloat16):
    """N(0, 1) with one percent of heavy-tailed (Student t, three degrees of freedom) entries."""
    x = torch.randn(rows, cols, generator=gen, device="cuda")
    chi2 = sum(torch.randn(rows, cols, generator=gen, device="cuda").square() for _ in range(3))
    heavy = torch.rand(rows, cols, generator=gen, device="cuda") < 0.01
    x = torch.where(heavy, torch.randn(rows, cols, generator=gen, device="cuda") / (chi2 / 3).sqrt(), x)
    return x.to(dtype)


def _layer(gen, case, scheme=PRODUCTION_SCHEME):
    hd = case["hd"]
    layer = q.QuantizedLinear(
        case["in"], case["out"], bias=False, device="cuda", dtype=torch.float32 if case.get("amp") else torch.bfloat16,
        weight_quantizer=q.QUANTIZER_CLASSES["QuestMXFP4Quantizer"](hadamard_dim=hd),
        activation_quantizer=q.QUANTIZER_CLASSES["QuestMXFP4Quantizer"](hadamard_dim=hd),
        gradient_quantizer=q.QUANTIZER_CLASSES["AlbertTsengQuantizer"](hadamard_dim=hd, stochastic=True, rerotate="signs"),
        backward_scheme=q.BACKWARD_SCHEMES[scheme]())
    with torch.no_grad():
        layer.weight.copy_(_normal(gen, case["out"], case["in"], scale=0.02, dtype=torch.float32))
    return layer


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    state = {"kind": kind, "seed": seed, "amp": bool(case.get("amp"))}
    if kind == "llama_eval":
        devices = [torch.cuda.current_device()]
        with torch.random.fork_rng(devices=devices), torch.device("cuda"):
            torch.manual_seed(seed)
            model = Llama(llama_30m()).eval()
        q.enable_packed_weight_cache(model)  # the weights do not change while the model is evaluated
        ids = torch.randint(0, model.config.vocab_size, (case["batch"], case["seq"] + 1), generator=gen, device="cuda")
        state.update(model=model, ids=ids[:, :-1].contiguous(), targets=ids[:, 1:].contiguous())
        return state
    T, I = case["tokens"], case["in"]
    if kind == "quantizer":
        cls = {"quest": "QuestMXFP4Quantizer", "albert": "AlbertTsengQuantizer"}[case["which"]]
        state.update(quantizer=q.QUANTIZER_CLASSES[cls](hadamard_dim=case["hd"]),
                     x=_activations(gen, T, I).requires_grad_(True), e=_normal(gen, T, I, scale=1e-3))
        return state
    layer = _layer(gen, case, ERROR_ONLY_SCHEME if kind == "error_only" else PRODUCTION_SCHEME)
    state["layer"] = layer
    if kind == "infer":
        q.enable_packed_weight_cache(layer)  # the weight does not change while the model serves
        state["x"] = _activations(gen, T, I)
        return state
    state["e"] = _normal(gen, T, case["out"], scale=1e-3)
    if kind == "norm_linear":
        norm = RMSNorm(I, eps=1e-5).to("cuda")
        with torch.no_grad():
            norm.weight.add_(_normal(gen, I, scale=0.1, dtype=torch.float32))
        state.update(norm=norm, x=_activations(gen, T, I, torch.float32).requires_grad_(True),
                     add=_normal(gen, T, I, scale=0.3).requires_grad_(True),
                     skip=_normal(gen, T, I, scale=1e-3, dtype=torch.float32))
    elif kind == "swiglu_linear":
        state["x"] = _activations(gen, T, 2 * I).requires_grad_(True)
    else:
        state["x"] = _activations(gen, T, I).requires_grad_(True)
    return state


def _seed(state):
    """Stochastic rounding draws its seeds and sign flips from the host generators: the same ones on every pass."""
    random.seed(state["seed"])
    torch.default_generator.manual_seed(state["seed"])


def run(state):
    kind = state["kind"]
    if kind == "infer":
        with torch.no_grad():
            return state["layer"](state["x"])
    if kind == "llama_eval":
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
            out = state["model"](state["ids"], targets=state["targets"], get_logits=True)
        return {"logits": out["logits"], "loss": out["loss"]}
    _seed(state)
    x = state["x"]
    x.grad = None
    if kind == "quantizer":
        y = state["quantizer"](x)
        y.backward(state["e"])
        return y, x.grad
    layer = state["layer"]
    layer.weight.grad = None
    if kind == "norm_linear":
        norm, add = state["norm"], state["add"]
        norm.weight.grad = add.grad = None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y, x_sum = rmsnorm_linear(norm, layer, x, pass_input=True, add=add)
            torch.autograd.backward([y, x_sum], [state["e"], state["skip"]])
        return y, x_sum, x.grad, add.grad, norm.weight.grad, layer.weight.grad
    if state["amp"]:
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = swiglu_linear(layer, x) if kind == "swiglu_linear" else layer(x)
            y.backward(state["e"])
    else:
        y = layer(x)
        y.backward(state["e"])
    return y, x.grad, layer.weight.grad


def work(case):
    kind = case["kind"]
    if kind == "llama_eval":
        cfg = llama_30m()
        tokens, d, f, v, n = case["batch"] * case["seq"], cfg.n_embd, cfg.ffn_dim, cfg.vocab_size, cfg.n_layer
        linear = n * (4 * d * d + 3 * d * f)
        # packed block weights, embedding rows, lm_head (fp32 master copy), logits out in bf16; causal attention's half square
        return {"bytes": linear * 17 / 32 + tokens * d * 4 + v * d * 4 + tokens * v * 2,
                "flops": 2.0 * tokens * (linear + v * d) + n * 2.0 * case["batch"] * case["seq"] ** 2 * d}
    T, I, O = case["tokens"], case["in"], case.get("out", 0)
    if kind == "quantizer":
        # x and e in, the quantized tensor and x's gradient out
        return {"bytes": 8.0 * T * I, "flops": 0.0}
    if kind == "infer":
        return {"bytes": 2.0 * T * I + O * I * 17 / 32 + 2.0 * T * O, "flops": 2.0 * T * I * O}
    weight = 4 if case["amp"] else 2
    layer = 2.0 * T * O * 2 + 2.0 * O * I * weight  # y, e; W and its gradient
    if kind == "norm_linear":
        # x (fp32), the summand and the skip gradient in; the sum, x's gradient (fp32) and the summand's out; the gain twice
        return {"bytes": layer + T * I * (4.0 + 2 + 4 + 4 + 4 + 2) + 8.0 * I, "flops": 6.0 * T * I * O}
    # x and its gradient (for SwiGLU both halves of the projection in front of it)
    return {"bytes": layer + 2.0 * T * I * 2 * (2 if kind == "swiglu_linear" else 1), "flops": 6.0 * T * I * O}


def tolerance(case):
    if case["kind"] == "quantizer":
        # an fp32 rotation summed in another order moves about one code in 10^4 to its neighbour, by up to half its value
        return {"rel": 1e-2, "max": 0.7}
    # bf16 results of fp32 accumulation
    return {"rel": 1e-2}
