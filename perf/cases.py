"""The calls that a Gemma 4 12B runtime makes on this library, for timing.

Every case goes through the package's public classes (``QuantizedLinear``,
``QuantizedGeGLU``, ``LoraAdapter``), with resident weights as a runtime keeps them.
The projections are those of the decoder that ``bench.py`` runs: hidden 3840, q|k|v as
one handle of 8192 rows, o 3840x4096, the gate|up pair of 15360 rows each, down
3840x15360, a tied embedding and head of 262144 rows; a full-attention layer has q of
8192 rows, k of 512 and o of 3840x8192.  Weights are N(0, 0.02) quantized by the
package's quantizer; activations are N(0, 1), with 1% of the entries scaled by 20 in
prompts.

Kinds of case:

* ``layer``: the projections of one decoder layer at `rows` rows.  Up to 16 rows (one
  token, or a block of drafted tokens to verify) it is replayed from a graph, as a
  decode loop does; longer ones (a prompt, or its tail) are called eagerly.
* ``head``: what one decoding step does on the tied embedding: the token's row
  gathered, and the greedy head with its logits.
* ``lora``: a layer's attention projections with an adapter on each of them.
* ``linear``: one projection, called eagerly.
"""

from __future__ import annotations

import math

import torch

from helios_amd import qmm
from helios_amd.quantize import quantize

HIDDEN, FFN, VOCAB, SOFTCAP = 3840, 15360, 262144, 30.0
GROUP = 64
# (name, N, K) of each kind of attention; the MLP is the same in both
ATTENTION = {
    "sliding": [("qkv", 8192, HIDDEN), ("o", HIDDEN, 4096)],
    "full": [("q", 8192, HIDDEN), ("k", 512, HIDDEN), ("o", HIDDEN, 8192)],
}
LORA = [("q", 4096, HIDDEN), ("k", 2048, HIDDEN), ("v", 2048, HIDDEN), ("o", HIDDEN, 4096)]


def listed():
    return [
        # the smallest call: one projection of one token, where the launch counts most
        {"name": "k_proj_1", "kind": "linear", "rows": 1, "n": 2048, "k": HIDDEN, "bits": 4, "dtype": "bf16"},
        # one token through a layer: the headline decode step
        {"name": "decode_layer_1", "kind": "layer", "rows": 1, "attn": "sliding", "bits": 4, "dtype": "bf16"},
        # a block of drafted tokens verified at once
        {"name": "verify_layer_8", "kind": "layer", "rows": 8, "attn": "sliding", "bits": 4, "dtype": "bf16"},
        # the 8-bit override, a short block
        {"name": "q8_verify_layer_3", "kind": "layer", "rows": 3, "attn": "sliding", "bits": 8, "dtype": "bf16"},
        # embedding gather and greedy head of one token, and of the longest verify block
        {"name": "token_head_1", "kind": "head", "rows": 1},
        {"name": "verify_head_16", "kind": "head", "rows": 16},
        # a short prompt, or the tail of a long one; a full-attention layer
        {"name": "prompt_full_layer_45", "kind": "layer", "rows": 45, "attn": "full", "bits": 4, "dtype": "bf16"},
        # an ordinary chat prompt
        {"name": "prompt_layer_200", "kind": "layer", "rows": 200, "attn": "sliding", "bits": 4, "dtype": "bf16"},
        # the float32 override, ragged rows
        {"name": "prompt_layer_517_f32", "kind": "layer", "rows": 517, "attn": "sliding", "bits": 4, "dtype": "f32"},
        # the 8-bit override in prefill
        {"name": "q8_prompt_layer_700", "kind": "layer", "rows": 700, "attn": "sliding", "bits": 8, "dtype": "bf16"},
        # adapters on q, k, v and o of a prompt
        {"name": "lora_attention_1100", "kind": "lora", "rows": 1100, "rank": 16},
        # one whole prefill chunk
        {"name": "prompt_layer_2048", "kind": "layer", "rows": 2048, "attn": "sliding", "bits": 4, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "prompt", "prompt", "head", "lora", "linear"])
    if kind == "decode":
        return {"kind": "layer", "rows": rng.randint(1, 16), "attn": rng.choice(["sliding", "full"]),
                "bits": rng.choice([4, 4, 8]), "dtype": "bf16"}
    if kind == "prompt":
        bits, dtype = rng.choice([(4, "bf16"), (4, "bf16"), (4, "f32"), (8, "bf16")])
        # an 8-bit layer, or one with float32 outputs, of 2048 rows would cost more than the largest listed case
        return {"kind": "layer", "rows": _log_int(rng, 17, 2048 if (bits, dtype) == (4, "bf16") else 1100),
                "attn": rng.choice(["sliding", "full"]), "bits": bits, "dtype": dtype}
    if kind == "head":
        return {"kind": "head", "rows": rng.randint(1, 16)}
    if kind == "lora":
        return {"kind": "lora", "rows": _log_int(rng, 1, 2048), "rank": rng.choice([4, 8, 16, 24, 32, 64])}
    return {"kind": "linear", "rows": _log_int(rng, 1, 2048), "n": _log_int(rng, 100, 16384),
            "k": GROUP * _log_int(rng, 4, 240), "bits": rng.choice([4, 4, 8]), "dtype": rng.choice(["bf16", "bf16", "f32"])}


class _Maker:
    """Inputs on the GPU from one seed; `triple` is what a checkpoint holds."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed) * 1000003 + 17)

    def randn(self, *shape):
        return torch.randn(shape, device="cuda", generator=self.g)

    def triple(self, n, k, bits):
        parts = [quantize((self.randn(min(32768, n - r), k) * 0.02).bfloat16(), GROUP, bits) for r in range(0, n, 32768)]
        return tuple(torch.cat(p) if len(parts) > 1 else p[0] for p in zip(*parts))

    def x(self, rows, k):
        x = self.randn(rows, k)
        if rows > 16:
            x = torch.where(torch.rand(x.shape, device="cuda", generator=self.g) < 0.01, x * 20, x)
        return x.bfloat16()


def _raw(case, seed):
    """The case's inputs as the checkpoint and the model hold them: weight triples by
    name, and the activations."""
    mk = _Maker(seed)
    rows, kind = case["rows"], case["kind"]
    if kind == "linear":
        return {"w": mk.triple(case["n"], case["k"], case["bits"])}, {"x": mk.x(rows, case["k"])}, {}
    if kind == "head":
        ids = torch.randint(0, VOCAB, (rows,), device="cuda", generator=mk.g, dtype=torch.int32)
        return {"lm": mk.triple(VOCAB, HIDDEN, 4)}, {"x": mk.x(rows, HIDDEN), "ids": ids}, {}
    if kind == "lora":
        w = {name: mk.triple(n, k, 4) for name, n, k in LORA}
        # kaiming-uniform A and a trained, small B; scale = alpha / rank with alpha = 2 rank
        ab = {name: ((torch.rand((case["rank"], k), device="cuda", generator=mk.g) * 2 - 1) / math.sqrt(k),
                     mk.randn(n, case["rank"]) * 0.02, 2.0) for name, n, k in LORA}
        return w, {"x": mk.x(rows, HIDDEN), "attn": mk.x(rows, 4096)}, ab
    w = {name: mk.triple(n, k, case["bits"]) for name, n, k in ATTENTION[case["attn"]]}
    for name, n, k in (("gate", FFN, HIDDEN), ("up", FFN, HIDDEN), ("down", HIDDEN, FFN)):
        w[name] = mk.triple(n, k, case["bits"])
    xs = {"x": mk.x(rows, HIDDEN), "attn": mk.x(rows, ATTENTION[case["attn"]][-1][2]), "x2": mk.x(rows, HIDDEN)}
    if case["dtype"] == "f32":
        xs["h"] = mk.x(rows, FFN)  # the model's bf16 h: down takes bf16 rows under the override, too
    return w, xs, {}


def _call(state):
    case, m, x = state["case"], state["mods"], state["x"]
    dtype = torch.float32 if case.get("dtype") == "f32" else torch.bfloat16
    kind = case["kind"]
    if kind == "linear":
        return {"y": m["w"](x["x"], out_dtype=dtype)}
    if kind == "head":
        row = m["lm"].embed(x["ids"])
        token, value, logits = m["lm"].forward_greedy(x["x"], softcap=SOFTCAP, return_logits=True)
        return {"row": row, "token": token, "value": value, "logits": logits}
    if kind == "lora":
        return {name: m[name].forward_lora(x["attn" if name == "o" else "x"], state["lora"][name]) for name, _, _ in LORA}
    out = {name: m[name](x["attn" if name == "o" else "x"], out_dtype=dtype) for name, _, _ in ATTENTION[case["attn"]]}
    if dtype is torch.float32:
        out["h"] = m["pair"](x["x2"], out_dtype=dtype)
        out["y"] = m["down"](x["h"], out_dtype=dtype)
    else:
        out["y"], out["h"] = m["pair"].forward_mlp(m["down"], x["x2"])
    return out


def prepare(case, seed):
    w, x, ab = _raw(case, seed)
    bits = case.get("bits", 4)
    mods = {name: qmm.QuantizedLinear(*t, group_size=GROUP, bits=bits) for name, t in w.items() if name not in ("gate", "up")}
    if "gate" in w:
        mods["pair"] = qmm.QuantizedGeGLU(w["gate"], w["up"], group_size=GROUP, bits=bits)
    lora = {name: qmm.LoraAdapter(a.cpu().numpy(), b.cpu().numpy(), scale) for name, (a, b, scale) in ab.items()}
    state = {"case": case, "mods": mods, "x": x, "lora": lora, "graph": None}
    if case["kind"] == "layer" and case["rows"] <= 16:
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _call(state)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            state["out"] = _call(state)
        state["graph"] = graph
    return state


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
        return state["out"]
    return _call(state)


def _weight_bytes(n, k, bits):
    return n * k * bits // 8 + 4 * n * (k // GROUP)


def work(case):
    m, kind = case["rows"], case["kind"]
    size = 4 if case.get("dtype") == "f32" else 2
    if kind == "linear":
        n, k = case["n"], case["k"]
        return {"bytes": _weight_bytes(n, k, case["bits"]) + 2 * m * k + size * m * n, "flops": 2 * m * n * k}
    if kind == "head":
        gather = m * (_weight_bytes(1, HIDDEN, 4) + 4 + 2 * HIDDEN)
        return {"bytes": _weight_bytes(VOCAB, HIDDEN, 4) + 2 * m * HIDDEN + m * (2 * VOCAB + 8) + gather,
                "flops": 2 * m * VOCAB * HIDDEN}
    if kind == "lora":
        r = case["rank"]
        return {"bytes": sum(_weight_bytes(n, k, 4) + 4 * r * (n + k) + 2 * m * n for _, n, k in LORA) + 2 * m * (HIDDEN + 4096),
                "flops": sum(2 * m * n * k + 2 * m * r * (n + k) for _, n, k in LORA)}
    attn = ATTENTION[case["attn"]]
    mats = attn + [("gate", FFN, HIDDEN), ("up", FFN, HIDDEN), ("down", HIDDEN, FFN)]
    io = 2 * m * (HIDDEN + attn[-1][2] + HIDDEN) + size * m * (sum(n for _, n, _ in attn) + FFN + HIDDEN)
    if size == 4:
        io += 2 * m * FFN
    return {"bytes": sum(_weight_bytes(n, k, case["bits"]) for _, n, k in mats) + io,
            "flops": sum(2 * m * n * k for _, n, k in mats)}


def tolerance(case):
    if case.get("dtype") == "f32":
        # 2e-5 (projections) and 1e-4 (the GeGLU's h) of the 64-bit results, measured; four times the larger
        return {"rel": 4e-4, "max": 4e-3}
    # bf16 outputs rounded once from 32-bit sums (GeGLU: after each of its operations): 2e-3 to 4e-3, measured
    out = {"rel": 1e-2, "max": 5e-2}
    if case["kind"] == "head":
        out["differ"] = 0.2
    return out


def _weight64(t, bits):
    w, s, b = t
    n, per = w.shape[0], 32 // bits
    codes = (w.view(torch.int32).unsqueeze(-1) >> torch.arange(0, 32, bits, device=w.device, dtype=torch.int32)) & (2 ** bits - 1)
    codes = codes.reshape(n, w.shape[1] * per // GROUP, GROUP)
    return (codes.double() * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).reshape(n, -1)


def _mm64(x, t, bits):
    x, n = x.double(), t[0].shape[0]
    return torch.cat([x @ _weight64(tuple(a[r:r + 16384] for a in t), bits).t() for r in range(0, n, 16384)], dim=1)


def _geglu64(g, u):
    # the model's bf16 constants
    return 0.5 * g * (1 + torch.tanh(0.796875 * (g + 0.044677734375 * g ** 3))) * u


def exact(case, seed):
    w, x, ab = _raw(case, seed)
    kind, bits = case["kind"], case.get("bits", 4)
    if kind == "linear":
        return {"y": _mm64(x["x"], w["w"], bits)}
    if kind == "head":
        row = _weight64(tuple(a[x["ids"].long()] for a in w["lm"]), 4)
        logits = torch.tanh(_mm64(x["x"], w["lm"], 4) / SOFTCAP) * SOFTCAP
        return {"row": row, "token": None, "value": logits.amax(dim=1), "logits": logits}
    if kind == "lora":
        out = {}
        for name, _, _ in LORA:
            xi = x["attn" if name == "o" else "x"]
            a, b, scale = ab[name]
            out[name] = _mm64(xi, w[name], 4) + (xi.double() @ a.double().t()) @ b.double().t() * scale
        return out
    out = {name: _mm64(x["attn" if name == "o" else "x"], w[name], bits) for name, _, _ in ATTENTION[case["attn"]]}
    out["h"] = _geglu64(_mm64(x["x2"], w["gate"], bits), _mm64(x["x2"], w["up"], bits))
    out["y"] = _mm64(x["h"] if "h" in x else out["h"], w["down"], bits)
    return out
