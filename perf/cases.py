"""The work that programs have this library do, as cases that can be timed and checked.

A case is one pass through a public entry point: ``OptimizedTransformer.forward``
(whole narrow models, and one-layer models of every other width), the attention
operator, the feed-forward operators and the residual-add + LayerNorm operator.
``listed`` holds the cases, ``draw`` gives further ones of the same ranges.

Sizes are those of the library's configurations (``tkmi/configs/baseline.json``
and ``shapes.json``) or generic ones beside them.
"""

from __future__ import annotations

import math
import pathlib
import sys

import torch
import torch.nn.functional as F

_PKG = str(pathlib.Path(__file__).resolve().parents[1] / "transformer-kernel_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import tkmi  # noqa: E402
from tkmi import ops  # noqa: E402

_DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
_EPS = 1e-5  # nn.LayerNorm's default

# Drawn cases stay below the largest listed ones: 4.4 Tflop each.
_MOST_FLOPS = 6e11
_MOST_BYTES = 1.5e9


def _model(name, batch, seq, d_model, heads, ffn, layers=1, causal=True, dtype="float32", padding=0.0):
    case = dict(kind="model", batch=batch, seq=seq, d_model=d_model, heads=heads, ffn=ffn, layers=layers,
                causal=causal, dtype=dtype, padding=padding)
    return dict(name=name, **case) if name else case


def _attention(name, batch, seq, heads, head_dim, causal, padding=0.0):
    case = dict(kind="attention", batch=batch, seq=seq, heads=heads, head_dim=head_dim, causal=causal,
                padding=padding)
    return dict(name=name, **case) if name else case


def _mlp(name, tokens, d_model, ffn):
    case = dict(kind="mlp", tokens=tokens, d_model=d_model, ffn=ffn)
    return dict(name=name, **case) if name else case


def _norm(name, rows, cols, y_dtype="float16", out_dtype="float16"):
    case = dict(kind="norm", rows=rows, cols=cols, y_dtype=y_dtype, out_dtype=out_dtype)
    return dict(name=name, **case) if name else case


def listed():
    return [
        # Whole forward of a narrow 4-layer model over a batch.
        _model("narrow_batch", 64, 128, 128, 4, 128, layers=4),
        # The smallest call: the same model on one sequence (appendix shape 2); latency and launches.
        _model("narrow_single", 1, 128, 128, 4, 128, layers=4),
        # A block over many short sequences, no causal mask.
        _model("block_short", 256, 64, 512, 8, 2048, causal=False),
        # A block on one prompt, in half precision, as a service runs it for one request.
        _model("block_single", 1, 512, 1024, 16, 4096, dtype="float16"),
        # An encoder block over a padded batch of an odd length.
        _model("block_padded", 6, 777, 768, 12, 3072, causal=False, padding=0.3),
        # A block with four 256-wide heads (appendix shape 8).
        _model("block_wide_heads", 64, 128, 1024, 4, 1024),
        # A narrow block over long sequences (appendix shape 13).
        _model("block_narrow_long", 64, 1024, 128, 4, 128),
        # The largest block.
        _model("block_large", 4, 8192, 2048, 16, 8192),
        # Causal attention over very long sequences.
        _attention("attention_long", 2, 32768, 16, 64, True),
        # Attention of an encoder: every query sees every key, 128-wide heads.
        _attention("attention_full", 4, 2048, 16, 128, False),
        # The feed-forward half of a block: GELU projection, residual projection.
        _mlp("mlp", 16384, 1024, 4096),
        # Residual add + LayerNorm of the same width, as a program that has its own projections calls it.
        _norm("norm", 16384, 1024),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _length(rng, lo, hi):
    """Half of the lengths are any whole number, the others multiples of 16, 64 or 128."""
    n = _log_int(rng, lo, hi)
    step = rng.choice((1, 1, 1, 16, 64, 128))
    return min(hi, max(lo, -(-n // step) * step))


def _draw_once(rng):
    kind = rng.choices(("narrow", "block", "attention", "mlp", "norm"), (2, 7, 3, 2, 1))[0]
    if kind == "narrow":
        return _model(None, _log_int(rng, 1, 512), _length(rng, 16, 128), 128, rng.choice((1, 2, 4, 8)), 128,
                      layers=rng.choice((2, 4, 6)), causal=rng.random() < 0.7)
    if kind == "block":
        head_dim = rng.choice((32, 64, 64, 64, 128, 128, 256, 80, 96))
        heads = rng.choice((2, 4, 8, 12, 16))
        d_model = heads * head_dim
        return _model(None, _log_int(rng, 1, 256), _length(rng, 16, 8192), d_model, heads,
                      d_model * rng.choice((1, 2, 4, 4)), causal=rng.random() < 0.6,
                      dtype=rng.choice(("float32", "float32", "float32", "float16", "bfloat16")),
                      padding=rng.choice((0.0, 0.0, 0.0, 0.3)))
    if kind == "attention":
        return _attention(None, _log_int(rng, 1, 128), _length(rng, 32, 32768), rng.choice((1, 2, 4, 8, 12, 16)),
                          rng.choice((32, 64, 64, 128, 128, 256)), rng.random() < 0.5,
                          padding=rng.choice((0.0, 0.0, 0.0, 0.3)))
    if kind == "mlp":
        d_model = rng.choice((256, 512, 640, 768, 1024, 1280, 1536, 2048))
        return _mlp(None, _length(rng, 32, 65536), d_model, d_model * rng.choice((1, 2, 4, 4)))
    return _norm(None, _length(rng, 64, 65536), rng.choice((128, 256, 512, 768, 1000, 1024, 2048, 4096)),
                 rng.choice(("float16", "float32")), rng.choice(("float16", "float32")))


def draw(rng):
    while True:
        case = _draw_once(rng)
        if case["kind"] == "model" and case["d_model"] > 2048:
            continue
        need = work(case)
        if need["flops"] <= _MOST_FLOPS and need["bytes"] <= _MOST_BYTES:
            return case


# --------------------------------------------------------------------------- #
# Inputs
# --------------------------------------------------------------------------- #


def _rand(gen, shape, std=1.0, mean=0.0):
    return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(mean, std, generator=gen)


def _linear_params(gen, out_features, in_features):
    """A projection's weight and bias, distributed as nn.Linear's default initialisation."""
    bound = 1.0 / math.sqrt(in_features)
    make = lambda *shape: torch.empty(shape, device="cuda").uniform_(-bound, bound, generator=gen)  # noqa: E731
    return make(out_features, in_features), make(out_features)


def _norm_params(gen, n):
    """LayerNorm weight and bias around their initial values, as training leaves them."""
    return _rand(gen, (n,), 0.1, 1.0), _rand(gen, (n,), 0.1)


def _lengths_mask(gen, batch, seq, padding):
    """[B, S] validity of a padded batch: lengths even over [(1 - padding) S, S], the longest one whole."""
    if padding <= 0:
        return None
    lo = max(1, int(seq * (1.0 - padding)))
    lengths = torch.randint(lo, seq + 1, (batch,), generator=gen, device="cuda")
    lengths[0] = seq
    if batch == 1:
        lengths[0] = lo
    return torch.arange(seq, device="cuda")[None, :] < lengths[:, None]


def _inputs(case, seed):
    """Tensors of a case, made from the seed alone; what `prepare` and `exact` both start from."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    kind = case["kind"]
    if kind == "model":
        dt = _DTYPES[case["dtype"]]
        d, f = case["d_model"], case["ffn"]
        params = {}
        for i in range(case["layers"]):
            p = f"layers.{i}."
            for n, (o, k) in (("attention.q_proj", (d, d)), ("attention.k_proj", (d, d)),
                              ("attention.v_proj", (d, d)), ("attention.out_proj", (d, d)), ("ffn_in", (f, d)),
                              ("ffn_out", (d, f))):
                params[p + n + ".weight"], params[p + n + ".bias"] = _linear_params(gen, o, k)
            for n in ("norm1", "norm2"):
                params[p + n + ".weight"], params[p + n + ".bias"] = _norm_params(gen, d)
        params["final_norm.weight"], params["final_norm.bias"] = _norm_params(gen, d)
        params = {k: v.to(dt) for k, v in params.items()}
        x = _rand(gen, (case["batch"], case["seq"], d)).to(dt)
        return {"params": params, "x": x, "mask": _lengths_mask(gen, case["batch"], case["seq"], case["padding"])}
    if kind == "attention":
        b, s, h, hd = case["batch"], case["seq"], case["heads"], case["head_dim"]
        qkv = torch.empty((b, s, 3, h, hd), dtype=torch.float16, device="cuda").normal_(generator=gen)
        return {"qkv": qkv, "mask": _lengths_mask(gen, b, s, case["padding"])}
    if kind == "mlp":
        t, d, f = case["tokens"], case["d_model"], case["ffn"]
        w1, b1 = _linear_params(gen, f, d)
        w2, b2 = _linear_params(gen, d, f)
        return {"h": _rand(gen, (t, d)).half(), "resid": _rand(gen, (t, d)), "w1": w1.half(), "b1": b1,
                "w2": w2.half(), "b2": b2}
    w, b = _norm_params(gen, case["cols"])
    return {"x": _rand(gen, (case["rows"], case["cols"])),
            "y": _rand(gen, (case["rows"], case["cols"]), 0.5).to(_DTYPES[case["y_dtype"]]), "w": w, "b": b}


def prepare(case, seed):
    state = _inputs(case, seed)
    state["case"] = case
    if case["kind"] == "model":
        config = tkmi.TransformerConfig(case["batch"], case["seq"], case["d_model"], case["heads"], case["ffn"],
                                        case["layers"], case["causal"])
        with torch.device("meta"):
            model = tkmi.OptimizedTransformer(config)
        model.load_state_dict(state.pop("params"), strict=True, assign=True)
        state["model"] = model.eval()
    elif case["kind"] == "attention":
        state["q"], state["k"], state["v"] = state.pop("qkv").permute(2, 0, 3, 1, 4).unbind(0)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    with torch.inference_mode():
        if kind == "model":
            return state["model"](state["x"], state["mask"])
        if kind == "attention":
            return ops.flash_attention(state["q"], state["k"], state["v"], case["head_dim"] ** -0.5, case["causal"],
                                       key_valid=state["mask"])
        if kind == "mlp":
            u = ops.linear(state["h"], state["w1"], state["b1"], gelu=True)
            return ops.linear_residual(u, state["w2"], state["b2"], state["resid"])
        return ops.add_ln_fwd(state["x"], state["y"], state["w"], state["b"], _EPS, _DTYPES[case["out_dtype"]])


# --------------------------------------------------------------------------- #
# What a pass cannot do without, and how far two correct ones can be apart
# --------------------------------------------------------------------------- #


def _attention_flops(case, head_dim):
    s = case["seq"]
    pairs = s * (s + 1) / 2 if case["causal"] else s * s
    if case["padding"]:
        # Lengths are even over [(1 - padding) S, S]: the mean of the valid keys (causal: of their pairs).
        keep = 1.0 - case["padding"] / 2
        pairs *= keep
    return 4.0 * case["batch"] * case["heads"] * head_dim * pairs


def work(case):
    kind = case["kind"]
    if kind == "model":
        t, d, f = case["batch"] * case["seq"], case["d_model"], case["ffn"]
        layer = 2.0 * t * (4 * d * d + 2 * d * f) + _attention_flops(case, d // case["heads"])
        elem = 4 if case["dtype"] == "float32" else 2
        weights = case["layers"] * (2.0 * (4 * d * d + 2 * d * f) + 4.0 * (9 * d + f))
        return {"bytes": 2.0 * elem * t * d + weights + (t if case["padding"] else 0),
                "flops": case["layers"] * layer}
    if kind == "attention":
        t, d = case["batch"] * case["seq"], case["heads"] * case["head_dim"]
        return {"bytes": 8.0 * t * d + (t if case["padding"] else 0), "flops": _attention_flops(case, case["head_dim"])}
    if kind == "mlp":
        t, d, f = case["tokens"], case["d_model"], case["ffn"]
        return {"bytes": t * d * (2.0 + 4 + 4) + 4.0 * d * f + 4.0 * (d + f), "flops": 4.0 * t * d * f}
    n = case["rows"] * case["cols"]
    size = lambda name: 4.0 if name == "float32" else 2.0  # noqa: E731
    return {"bytes": n * (8.0 + size(case["y_dtype"]) + size(case["out_dtype"])) + 8.0 * case["cols"], "flops": 8.0 * n}


def tolerance(case):
    """About four times what the results were seen to differ from 64 bits (fp16 operands, fp32 sums)."""
    kind = case["kind"]
    if kind == "model":
        if case["dtype"] == "bfloat16":  # 1.7e-3: the rounding of the output
            return {"rel": 7e-3, "max": 2e-2}
        if case["dtype"] == "float16" or case["layers"] > 1:  # 2.2e-4: output rounding; 2.5e-4 over six layers
            return {"rel": 1e-3, "max": 6e-3}
        return {"rel": 4e-4, "max": 4e-3}  # 9.5e-5, largest 7.4e-4
    if kind == "attention":  # 2.9e-4, largest 1.0e-2 where an average over many keys is near 0
        return {"rel": 1.2e-3, "max": 4e-2}
    if kind == "mlp":  # 4.1e-5, largest 2.2e-4
        return {"rel": 2e-4, "max": 1e-3}
    if case["out_dtype"] == "float16":  # 2.1e-4, largest 4.9e-4: the rounding of the output
        return {"rel": 8e-4, "max": 2e-3}
    return {"rel": 5e-7, "max": 5e-6}  # 6.5e-8, largest 3.4e-7


# --------------------------------------------------------------------------- #
# The same in 64 bits
# --------------------------------------------------------------------------- #


def _exact_attention(q, k, v, scale, causal, mask):
    """[B, S, H*hd] of [B, H, S, hd] operands; scores in pieces of at most 2^27 values."""
    b, h, s, hd = q.shape
    out = torch.empty((b, s, h, hd), dtype=torch.float64, device=q.device)
    keys = torch.arange(s, device=q.device)
    rows = max(1, min(s, 2 ** 27 // s))
    heads = max(1, min(h, 2 ** 27 // (rows * s)))
    for i in range(b):
        for j in range(0, h, heads):
            kt = k[i, j:j + heads].double().transpose(1, 2).contiguous()
            vj = v[i, j:j + heads].double().contiguous()
            for r in range(0, s, rows):
                e = min(s, r + rows)
                # A causal piece needs the keys up to its last row only.
                n = e if causal else s
                sc = torch.bmm(q[i, j:j + heads, r:e].double().contiguous(), kt[:, :, :n].contiguous()) * scale
                if causal:
                    sc.masked_fill_(keys[None, None, :n] > keys[None, r:e, None], -math.inf)
                if mask is not None:
                    sc.masked_fill_(~mask[i, None, None, :n], -math.inf)
                p = torch.softmax(sc, -1)
                out[i, r:e, j:j + heads] = torch.bmm(p, vj[:, :n].contiguous()).transpose(0, 1)
    return out.view(b, s, h * hd)


def _exact_model(case, seed):
    inp = _inputs(case, seed)
    w = {k: v.double() for k, v in inp["params"].items()}
    x, mask = inp["x"].double(), inp["mask"]
    b, s, d = x.shape
    h = case["heads"]
    gone = None if mask is None else ~mask[:, :, None]

    def norm(t, n):
        return F.layer_norm(t, (d,), w[n + ".weight"], w[n + ".bias"], _EPS)

    def lin(t, n):
        return torch.addmm(w[n + ".bias"], t.reshape(b * s, -1), w[n + ".weight"].t()).view(b, s, -1)

    for i in range(case["layers"]):
        p = f"layers.{i}."
        y = norm(x, p + "norm1")
        q, k, v = (lin(y, p + f"attention.{n}_proj").view(b, s, h, d // h).transpose(1, 2) for n in "qkv")
        a = lin(_exact_attention(q, k, v, (d // h) ** -0.5, case["causal"], mask), p + "attention.out_proj")
        del q, k, v
        x = x + (a if gone is None else a.masked_fill(gone, 0.0))
        x = x + lin(F.gelu(lin(norm(x, p + "norm2"), p + "ffn_in")), p + "ffn_out")
        if gone is not None:
            x = x.masked_fill(gone, 0.0)
    x = norm(x, "final_norm")
    return x if gone is None else x.masked_fill(gone, 0.0)


def exact(case, seed):
    kind = case["kind"]
    with torch.inference_mode():
        if kind == "model":
            return _exact_model(case, seed)
        inp = _inputs(case, seed)
        if kind == "attention":
            q, k, v = inp["qkv"].permute(2, 0, 3, 1, 4).unbind(0)
            return _exact_attention(q, k, v, case["head_dim"] ** -0.5, case["causal"], inp["mask"])
        d = {n: t.double() for n, t in inp.items()}
        if kind == "mlp":
            u = F.gelu(torch.addmm(d["b1"], d["h"], d["w1"].t()))
            return torch.addmm(d["b2"], u, d["w2"].t()) + d["resid"]
        s = d["x"] + d["y"]
        return s, F.layer_norm(s, (case["cols"],), d["w"], d["b"], _EPS)
