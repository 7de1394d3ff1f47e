"""Performance cases of the Q4 matrix-product path, through its public entry
points (marlin-mlx_amd/__init__.py).

What a program of this framework does, and the cases that stand for it:

  proj_*    one quantized product (qmatmul): the attention / SSM projections,
            for one token, for a few concurrent streams, for a short prompt
            and for a video turn's prompt
  mlp_*     one decoder block's MLP half (mlp_residual) over a prompt
  rows_*    the MLP halves of all layers for a batch of decode streams
            (BatchedMlpLayers)
  head_*    final norm + lm_head + greedy token with its logits
            (lm_head_argmax)
  step_*    one whole greedy decode step in one launch (DecodeStep)
  sample_*  temperature / top-k / top-p sampling of a logits row
            (sample_token)
  pack_*    quantizing the weights of a checkpoint shard (quantize_weights)

Sizes: hidden 2048, intermediate 6144, 24 layers and 248,320 vocabulary rows
are the configuration that the tests and the benchmark use; 512 / 2048 / 4096 /
6144 are its projection widths; 1960 tokens are a 10-frame video turn.

Weights are normal with sigma 0.02 in MLX's affine 4-bit layout, formed by
`_affine` in plain torch, so that `exact` needs none of the framework's code.
Activations are normal with a spread of channel scales.
"""
from __future__ import annotations

import importlib
import math

import torch

mq4 = importlib.import_module("marlin-mlx_amd")

HIDDEN, INTER, LAYERS, VOCAB = 2048, 6144, 24, 248320
SHARD = 6                    # layers of one checkpoint shard
EPS = 1e-6
Q4_BYTES = 0.5625            # per weight: a nibble, and a bf16 scale and bias per 64


# ------------------------------------------------------------------ cases ---

def listed() -> list[dict]:
    return [
        # the smallest call: one token's key or value projection
        {"name": "proj_token", "kind": "proj", "m": 1, "n": 512, "k": HIDDEN},
        # seven concurrent streams through a query projection
        {"name": "proj_rows", "kind": "proj", "m": 7, "n": 4096, "k": HIDDEN},
        # a one-sentence prompt through a projection
        {"name": "proj_prompt_short", "kind": "proj", "m": 77, "n": 4096, "k": HIDDEN},
        # a video turn's prompt through the widest projection
        {"name": "proj_prompt", "kind": "proj", "m": 1960, "n": 6144, "k": HIDDEN},
        # a short chat turn's prompt, an odd number of rows
        {"name": "mlp_prompt_short", "kind": "mlp", "m": 203, "h": HIDDEN, "i": INTER},
        # a video turn's prompt
        {"name": "mlp_prompt", "kind": "mlp", "m": 1960, "h": HIDDEN, "i": INTER},
        # a long prompt
        {"name": "mlp_prompt_long", "kind": "mlp", "m": 8192, "h": HIDDEN, "i": INTER},
        # one decode step's MLP halves for 16 concurrent streams
        {"name": "rows_stack", "kind": "rows", "m": 16, "layers": LAYERS},
        # the same step's lm_head
        {"name": "head_rows", "kind": "head", "m": 16, "v": VOCAB},
        # one stream's decode step
        {"name": "step_token", "kind": "step", "layers": LAYERS, "v": VOCAB},
        # a stochastic token of one stream with both filters on
        {"name": "sample_token", "kind": "sample", "m": 1, "v": VOCAB, "temperature": 0.7, "top_k": 50,
         "top_p": 0.9},
        # the loader: one checkpoint shard, six layers' matrices and the lm_head
        {"name": "pack_shard", "kind": "pack", "layers": SHARD, "v": VOCAB},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    """An integer of [lo, hi], spread evenly over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["proj", "proj", "mlp", "mlp", "rows", "head", "step", "sample", "pack"])
    if kind == "proj":
        # mostly the model's widths, else any width (a shard or a head of one)
        n = rng.choice([512, 2048, 4096, 6144]) if rng.random() < 0.7 else _log_int(rng, 128, 6144)
        return {"kind": kind, "m": _log_int(rng, 1, 2048), "n": n, "k": rng.choice([HIDDEN, HIDDEN, 1024, INTER])}
    if kind == "mlp":
        h, i = (HIDDEN, INTER) if rng.random() < 0.7 else (1024, 3072)
        return {"kind": kind, "m": _log_int(rng, 33, 8192), "h": h, "i": i}
    if kind == "rows":
        return {"kind": kind, "m": _log_int(rng, 1, 32), "layers": rng.randint(2, LAYERS)}
    if kind == "head":
        return {"kind": kind, "m": _log_int(rng, 1, 32), "v": _log_int(rng, 32000, VOCAB)}
    if kind == "step":
        return {"kind": kind, "layers": rng.randint(2, LAYERS), "v": _log_int(rng, 32000, VOCAB)}
    if kind == "sample":
        return {"kind": kind, "m": _log_int(rng, 1, 32), "v": _log_int(rng, 32000, VOCAB),
                "temperature": round(rng.uniform(0.3, 1.3), 2), "top_k": rng.choice([0, 20, 50, 200]),
                "top_p": rng.choice([0.5, 0.9, 0.95, 1.0])}
    return {"kind": kind, "layers": rng.randint(1, SHARD), "v": _log_int(rng, 32000, VOCAB)}


# ----------------------------------------------------------------- inputs ---

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g: torch.Generator, *shape: int, sigma: float = 1.0) -> torch.Tensor:
    return torch.randn(shape, generator=g, device="cuda") * sigma


def _acts(g: torch.Generator, m: int, k: int) -> torch.Tensor:
    """bf16 activations [m, k]: normal, the channels' scales spread log-normally."""
    return (_normal(g, m, k) * torch.exp(_normal(g, 1, k, sigma=0.5))).to(torch.bfloat16)


def _norm_weight(g: torch.Generator, k: int) -> torch.Tensor:
    return _normal(g, k, sigma=0.1).to(torch.bfloat16)


def _affine(w: torch.Tensor):
    """MLX's affine 4-bit, group-64 form of bf16 w [n, k], in float32: packed
    words int32 [n, k / 8] (low nibble first), bf16 scales and biases
    [n, k / 64]."""
    n, k = w.shape
    v = w.float().view(n, k // 64, 64)
    lo, hi = v.amin(-1, keepdim=True), v.amax(-1, keepdim=True)
    scale = ((hi - lo) / 15).clamp_min(1e-7)
    low = lo.abs() > hi.abs()
    scale = torch.where(low, scale, -scale)
    edge = torch.where(low, lo, hi)
    q0 = torch.round(edge / scale)
    some = q0 != 0
    scale = torch.where(some, edge / torch.where(some, q0, torch.ones_like(q0)), scale)
    bias = torch.where(some, edge, torch.zeros_like(edge))
    q = torch.round((v - bias) / scale).clamp_(0, 15).to(torch.int32).view(n, k // 8, 8)
    words = torch.zeros((n, k // 8), dtype=torch.int32, device=w.device)
    for p in range(8):
        words |= q[:, :, p] << (4 * p)
    return words, scale.view(n, -1).to(torch.bfloat16), bias.view(n, -1).to(torch.bfloat16)


def _weight(g: torch.Generator, n: int, k: int):
    return _affine(_normal(g, n, k, sigma=0.02).to(torch.bfloat16))


def _mlp(g: torch.Generator, h: int, i: int) -> dict:
    return {"norm": _norm_weight(g, h), "gate": _weight(g, i, h), "up": _weight(g, i, h), "down": _weight(g, h, i)}


def _inputs(case: dict, seed: int) -> dict:
    """The tensors of a case, before they are wrapped in the framework's types."""
    g, kind = _gen(seed), case["kind"]
    if kind == "proj":
        return {"x": _acts(g, case["m"], case["k"]), "w": _weight(g, case["n"], case["k"])}
    if kind == "mlp":
        return {"x": _acts(g, case["m"], case["h"]), "mlp": _mlp(g, case["h"], case["i"])}
    if kind == "rows":
        return {"x": _acts(g, case["m"], HIDDEN), "stack": [_mlp(g, HIDDEN, INTER) for _ in range(case["layers"])]}
    if kind == "head":
        return {"x": _acts(g, case["m"], HIDDEN), "norm": _norm_weight(g, HIDDEN), "w": _weight(g, case["v"], HIDDEN)}
    if kind == "step":
        return {"x": _acts(g, 1, HIDDEN), "stack": [_mlp(g, HIDDEN, INTER) for _ in range(case["layers"])],
                "norm": _norm_weight(g, HIDDEN), "w": _weight(g, case["v"], HIDDEN)}
    if kind == "sample":
        # a few clear candidates above a broad background
        m, v = case["m"], case["v"]
        logits = _normal(g, m, v, sigma=2.5)
        at = torch.randint(0, v, (m, 12), generator=g, device="cuda")
        logits.scatter_add_(1, at, 8.0 + _normal(g, m, 12, sigma=2.0))
        return {"logits": logits.to(torch.bfloat16), "seed": seed}
    ws = []
    for _ in range(case["layers"]):
        for n, k in ((INTER, HIDDEN), (INTER, HIDDEN), (HIDDEN, INTER)):
            ws.append(_normal(g, n, k, sigma=0.02).to(torch.bfloat16))
    ws.append(_normal(g, case["v"], HIDDEN, sigma=0.02).to(torch.bfloat16))
    return {"ws": ws}


def _qt(w) -> "mq4.QuantizedTensor":
    return mq4.QuantizedTensor(*w)


def _weights(m: dict) -> "mq4.MLPWeights":
    return mq4.MLPWeights(_qt(m["gate"]), _qt(m["up"]), _qt(m["down"]))


def _layers(stack: list[dict]) -> list:
    return [mq4.DecoderLayer(m["norm"], _weights(m)) for m in stack]


def prepare(case: dict, seed: int) -> dict:
    """What a program holds before the call: the activations, the quantized
    weights, and for the stacked entry points the object that keeps the layer
    table and its workspace."""
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "proj":
        return {"kind": kind, "x": t["x"], "w": _qt(t["w"])}
    if kind == "mlp":
        return {"kind": kind, "x": t["x"], "norm": t["mlp"]["norm"], "mlp": _weights(t["mlp"])}
    if kind == "rows":
        return {"kind": kind, "x": t["x"], "plan": mq4.BatchedMlpLayers(_layers(t["stack"]), case["m"], EPS)}
    if kind == "head":
        return {"kind": kind, "x": t["x"], "norm": t["norm"], "w": _qt(t["w"])}
    if kind == "step":
        return {"kind": kind, "x": t["x"], "plan": mq4.DecodeStep(_layers(t["stack"]), t["norm"], _qt(t["w"]), EPS),
                "x_out": torch.empty_like(t["x"])}
    if kind == "sample":
        return {"kind": kind, "logits": t["logits"], "temperature": case["temperature"], "top_k": case["top_k"],
                "top_p": case["top_p"], "seed": t["seed"]}
    return {"kind": kind, "ws": t["ws"]}


def run(state: dict):
    kind = state["kind"]
    if kind == "proj":
        return mq4.qmatmul(state["x"], state["w"])
    if kind == "mlp":
        return mq4.mlp_residual(state["x"], state["mlp"], state["norm"], EPS)
    if kind == "rows":
        return state["plan"](state["x"])
    if kind == "head":
        return mq4.lm_head_argmax(state["x"], state["w"], return_logits=True, norm_weight=state["norm"], eps=EPS)
    if kind == "step":
        token = state["plan"](state["x"], x_out=state["x_out"])
        return token, state["x_out"]
    if kind == "sample":
        return mq4.sample_token(state["logits"], state["temperature"], state["top_k"], state["top_p"],
                                seed=state["seed"])
    return [(q.weight, q.scales, q.biases) for q in mq4.quantize_weights(state["ws"])]


# -------------------------------------------------------- work, tolerance ---

def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "proj":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": Q4_BYTES * n * k + 2 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "mlp":
        m, h, i = case["m"], case["h"], case["i"]
        return {"bytes": Q4_BYTES * 3 * h * i + 2 * h + 4 * m * h, "flops": 6 * m * h * i}
    if kind == "rows":
        m, n = case["m"], case["layers"]
        return {"bytes": n * (Q4_BYTES * 3 * HIDDEN * INTER + 2 * HIDDEN) + 4 * m * HIDDEN,
                "flops": n * 6 * m * HIDDEN * INTER}
    if kind == "head":
        m, v = case["m"], case["v"]
        return {"bytes": Q4_BYTES * v * HIDDEN + 2 * HIDDEN + 2 * m * HIDDEN + 2 * m * v + 4 * m,
                "flops": 2 * m * v * HIDDEN}
    if kind == "step":
        n, v = case["layers"], case["v"]
        return {"bytes": n * (Q4_BYTES * 3 * HIDDEN * INTER + 2 * HIDDEN) + Q4_BYTES * v * HIDDEN + 6 * HIDDEN + 4,
                "flops": n * 6 * HIDDEN * INTER + 2 * v * HIDDEN}
    if kind == "sample":
        m, v = case["m"], case["v"]
        return {"bytes": 2 * m * v + 8 * m, "flops": 0}
    count = case["layers"] * 3 * HIDDEN * INTER + case["v"] * HIDDEN
    return {"bytes": (2 + Q4_BYTES) * count, "flops": 0}


def tolerance(case: dict):
    kind = case["kind"]
    if kind in ("sample", "pack"):
        return "exact"               # codes, scales, biases and tokens are defined to the bit
    # Measured against `exact`: 1.7e-3 (2-norm) for one product, the rounding of
    # its bf16 result; 2.3e-3 for the lm_head (its normalized input is bf16
    # too); 3.0e-3 for an MLP half (three more bf16 roundings on the way);
    # 1.8e-2 after 24 of them.  Two implementations share most roundings, so
    # between them less.  "max" counts units of 2^-8 in the same way.
    if kind == "proj":
        return {"rel": 3e-3, "max": 1.6e-2}
    if kind == "head":
        return {"rel": 5e-3, "max": 4e-2, "differ": 0.05}     # a token: at a tie of the two largest logits
    if kind == "mlp":
        return {"rel": 6e-3, "max": 6e-2}
    return {"rel": 5e-2, "max": 0.3, "differ": 0.05}


# ------------------------------------------------------------------ exact ---

def _dense(w) -> torch.Tensor:
    """The float64 matrix [n, k] that packed words, scales and biases stand for."""
    words, s, b = w
    n, k = words.shape[0], words.shape[1] * 8
    q = torch.stack([(words >> (4 * p)) & 15 for p in range(8)], dim=-1).view(n, k // 64, 64)
    return (q.double() * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).view(n, k)


def _rms_norm(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * (1 + w.double())


def _mlp_exact(x: torch.Tensor, m: dict) -> torch.Tensor:
    n = _rms_norm(x, m["norm"])
    g = n @ _dense(m["gate"]).t()
    u = n @ _dense(m["up"]).t()
    return x + (torch.sigmoid(g) * g * u) @ _dense(m["down"]).t()


def exact(case: dict, seed: int):
    """What run returns, in 64 bits without any rounding between the ops."""
    kind = case["kind"]
    if kind in ("sample", "pack"):
        return None                  # compared bit for bit
    t = _inputs(case, seed)
    x = t["x"].double()
    if kind == "proj":
        return x @ _dense(t["w"]).t()
    if kind == "mlp":
        return _mlp_exact(x, t["mlp"])
    if kind == "head":
        return None, _rms_norm(x, t["norm"]) @ _dense(t["w"]).t()
    for m in t["stack"]:
        x = _mlp_exact(x, m)
    return x if kind == "rows" else (None, x)
