"""The calls whose time matters to a program that uses this package, for measuring it.

``listed()`` are twelve of them at fixed sizes, ``draw(rng)`` gives further ones of the same ranges.  Models are the
configurations of ``bench.py`` (``chatrwkv_amd.synth.SHAPES``), one generic RWKV-5.2 model, and, among the drawn
cases, models of other depths and widths.  Weights are random, with the distributions of ``chatrwkv_amd.synth``;
every model has all of its layers.

Kinds:
  decode   one generated token: ``model.forward([id], state)`` in the middle of a reply.  Bound by the weights.
  prefill  one call with a prompt or a piece of one: ``model.forward(ids, state)``, the state carried on; with
           ``full`` the logits of every position (scoring a text).
  sample   the draw after a forward: penalties, nucleus, one id (``chatrwkv_amd.sampling.Sampler``).
  mm8      the uint8 product alone, as block code that calls the operators directly has it (``chatrwkv_amd.ops.mm8``).
"""
import math

import torch

from chatrwkv_amd import ops, synth
from chatrwkv_amd.model import RWKV
from chatrwkv_amd.model_v7 import RWKV_x070
from chatrwkv_amd.sampling import Sampler

# version, layers, width, channel-mix width, vocabulary
MODELS = {name: shape for name, shape in synth.SHAPES.items()}
MODELS["v5-1b5"] = (5.2, 24, 2048, 7168, 65536)

LORA_MAA, LORA_DECAY = 32, 64       # RWKV-6 ranks (the defaults of synth.make_checkpoint)
LOW, HIGH = 2, 2048                 # tokens of the shortest and of the longest sequence call
MOST = 5.5e12                       # values of weights times tokens that a drawn call stays under


def _model(name, strategy):
    version, layers, width, ffn, vocab = MODELS[name]
    return {"version": version, "layers": layers, "width": width, "ffn": ffn, "vocab": vocab, "strategy": strategy}


def listed():
    return [
        # A reply's next token on the three large models people chat with: int8 weights where the format has them.
        {"name": "decode_v4_7b_u8", "kind": "decode", **_model("v4-7b", "cuda fp16i8")},
        {"name": "decode_v6_7b_u8", "kind": "decode", **_model("v6-7b", "cuda fp16i8")},
        {"name": "decode_v7_7b_f16", "kind": "decode", **_model("v7-7b", "cuda fp16")},
        # The same on a model so small that launches, not bytes, are the time.
        {"name": "decode_v4_169m_f16", "kind": "decode", **_model("v4-169m", "cuda fp16")},
        # A long prompt in one call.
        {"name": "prompt_v4_7b_u8", "kind": "prefill", **_model("v4-7b", "cuda fp16i8"), "tokens": 1024, "full": False},
        # What a person types: one turn of a chat.
        {"name": "turn_v4_7b_u8", "kind": "prefill", **_model("v4-7b", "cuda fp16i8"), "tokens": 45, "full": False},
        # A prompt in pieces of 256, the chunk length of the chat programs: one such piece.
        {"name": "chunk_v6_7b_u8", "kind": "prefill", **_model("v6-7b", "cuda fp16i8"), "tokens": 256, "full": False},
        # A prompt of no particular length, unquantised.
        {"name": "prompt_v7_7b_f16", "kind": "prefill", **_model("v7-7b", "cuda fp16"), "tokens": 777, "full": False},
        {"name": "prompt_v5_1b5_f16", "kind": "prefill", **_model("v5-1b5", "cuda fp16"), "tokens": 333, "full": False},
        # Scoring a text: the logits of every position (vocabulary 50277, an odd width).
        {"name": "score_v4_169m_f16", "kind": "prefill", **_model("v4-169m", "cuda fp16"), "tokens": 513, "full": True},
        # The draw of a chat reply.
        {"name": "sample_65536", "kind": "sample", "vocab": 65536, "top_p": 0.7, "top_k": 0},
        # The widest product of the 7B models by itself.
        {"name": "mm8_1024_4096_16384", "kind": "mm8", "rows": 1024, "n": 4096, "m": 16384},
    ]


def draw(rng):
    kind = rng.choices(["prefill", "decode", "mm8", "sample"], [6, 2, 2, 1])[0]
    if kind == "sample":
        return {"kind": kind, "vocab": rng.choice([50277, 65536, rng.randint(20000, 65536)]),
                "top_p": round(rng.uniform(0.3, 0.95), 3), "top_k": rng.choice([0, 0, rng.randint(20, 200)])}
    if kind == "mm8":
        n = rng.choice([768, 2048, 4096, 5120])
        n, m = rng.choice([(n, n), (n, 4 * n), (4 * n, n)])
        return {"kind": kind, "rows": _log(rng, 1, HIGH if n * m < 1e8 else HIGH // 2), "n": n, "m": m}
    if rng.random() < 0.4:
        name = rng.choice(list(MODELS))
        case = _model(name, "cuda fp16" if MODELS[name][0] == 7 else rng.choice(["cuda fp16i8", "cuda fp16"]))
    else:
        version, width = rng.choice([4, 5.2, 6, 7]), 128 * _log(rng, 4, 32)
        ffn = 4 * width if version in (4, 7) else (width * 7 // 2) // 64 * 64
        case = {"version": version, "layers": rng.randint(6, 32), "width": width, "ffn": ffn, "vocab": rng.choice([50277, 65536]),
                "strategy": "cuda fp16" if version == 7 else rng.choice(["cuda fp16i8", "cuda fp16"])}
    case["kind"] = kind
    if kind == "prefill":
        case["full"] = rng.random() < 0.2
        values = sum(_matrix_values(case)) + case["width"] * case["vocab"]
        case["tokens"] = _log(rng, LOW, max(LOW, min(HIGH // 2 if case["full"] else HIGH, int(MOST / values))))
    return case


def _log(rng, low, high):
    """A whole number of [low, high], evenly spread over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))))


def _build(case, seed):
    shape = {"n_layer": case["layers"], "n_embd": case["width"], "n_ffn": case["ffn"], "vocab": case["vocab"], "seed": seed,
             "device": "cuda"}
    if case["version"] == 7:
        w = synth.make_checkpoint_v7(**shape)
        # The spreads of the other formats' matrices (0.02, LoRA first stages 0.01): with its own larger ones a model of
        # all its layers blows the last bit of a rounding up to several percent of its logits, as no trained model does.
        for k, t in w.items():
            if k.endswith(("receptance.weight", "key.weight", "value.weight", "output.weight")):
                t.mul_(0.02 / 0.05)
            elif k.endswith(("att.w1", "att.a1", "att.v1", "att.g1")):
                t.mul_(0.01 / 0.1)
            elif k.endswith(("att.w2", "att.a2", "att.v2", "att.g2")):
                t.mul_(0.1 / 0.2)
        return RWKV_x070(w, case["strategy"])
    return RWKV(synth.make_checkpoint(version=case["version"], lora_maa=LORA_MAA, lora_decay=LORA_DECAY, **shape),
                case["strategy"], verbose=False)


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    if case["kind"] == "sample":
        V = case["vocab"]
        # logits of a trained model: a few dozen likely ids, the rest far below; eight ids drawn so far
        logits = torch.randn(V, generator=g, device="cuda") * 3.0
        s = Sampler(V, token_ban=[0], seed=int(seed))
        for i in torch.randint(0, V, (8,), generator=g, device="cuda").tolist():
            row = torch.full((V,), -20.0, device="cuda")
            row[i] = 20.0
            s.sample(row, u=0.5, alpha_decay=0.996)
        u = torch.rand(1, generator=g, device="cuda")
        return {"case": case, "sampler": s, "logits": logits, "u": u}
    if case["kind"] == "mm8":
        w = torch.randn((case["m"], case["n"]), generator=g, device="cuda") * 0.02
        q = ops.quantize_u8(w.t(), scale_dtype=torch.float16, input_contiguous=True)
        rows = case["rows"]
        x = torch.randn((rows, case["n"]) if rows > 1 else (case["n"],), generator=g, device="cuda").half()
        return {"case": case, "x": x, "w": q}
    model = _build(case, seed)
    ids = synth.random_tokens(16 + max(16, case.get("tokens", 0)), case["vocab"], seed=seed)
    # the conversation so far, and the first token of the reply
    _, state = model.forward(ids[:15], None)
    if case["kind"] == "decode":
        _, state = model.forward([ids[15]], state)
    return {"case": case, "model": model, "state": state, "ids": ids[16:], "next": 0}


def run(state):
    case = state["case"]
    if case["kind"] == "sample":
        s = state["sampler"]
        token = s.sample(state["logits"], temperature=1.0, top_p=case["top_p"], top_k=case["top_k"], alpha_presence=0.2,
                         alpha_frequency=0.2, alpha_decay=0.996, u=state["u"])
        return {"token": token, "probs": s.probs, "occurrence": s.occurrence, "seen": s.seen}
    if case["kind"] == "mm8":
        return ops.mm8(state["x"], *state["w"])
    if case["kind"] == "decode":
        ids = [state["ids"][state["next"] % len(state["ids"])]]
        state["next"] += 1
        out, st = state["model"].forward(ids, state["state"])
    else:
        out, st = state["model"].forward(state["ids"][:case["tokens"]], state["state"], full_output=case["full"])
    # every tensor of the state is a piece of these two
    return {"logits": out, "state16": st.flat[0], "state32": st.flat[1]}


def _matrix_values(case):
    """Weights of the large matrices and of the LoRA pairs, without the head."""
    version, layers, width = case["version"], case["layers"], case["width"]
    square = {4: 4 + 1, 5.2: 5 + 1, 6: 5 + 1, 7: 4}[version]
    big = layers * (square * width * width + 2 * width * case["ffn"])
    lora = 0
    if version == 6:
        lora = layers * width * 2 * (5 * LORA_MAA + LORA_DECAY)
    elif version == 7:
        lora = layers * width * 2 * sum(synth.v7_lora_dims(width))
    return big, lora


def work(case):
    if case["kind"] == "sample":
        V = case["vocab"]
        return {"bytes": 4 * V + 4 * V + 2 * 4 * V + 2 * V, "flops": 40 * V}   # logits, probabilities, both tables updated
    if case["kind"] == "mm8":
        b, n, m = case["rows"], case["n"], case["m"]
        return {"bytes": n * m + 2 * b * (n + m) + 4 * (n + m), "flops": 2 * b * n * m}
    version, layers, width, vocab = case["version"], case["layers"], case["width"], case["vocab"]
    tokens = case.get("tokens", 1)
    rows = tokens if case.get("full") else 1                           # rows that go through the head
    big, lora = _matrix_values(case)
    head = width * vocab
    each = 1 if "i8" in case["strategy"] else 2
    per_head = 0 if version == 4 else 64
    state = layers * (2 * width * 2 + (3 * width * 4 if version == 4 else width * per_head * 4))
    logits = rows * vocab * (2 if version == 7 else 4)
    recurrence = layers * width * (12 if version == 4 else (6 if version < 7 else 8) * per_head)
    return {"bytes": (big + head) * each + lora * 2 + tokens * width * 2 + 2 * state + logits,
            "flops": 2 * tokens * (big + lora) + 2 * rows * head + tokens * recurrence}


# Four times what full-depth models differ by from themselves when their sums are taken in another order (a prompt in
# one call and in two, other tiles, other splits): rel 3.3e-3 / 4.1e-3 / 6.5e-3 / 6.8e-3, largest 0.016 / 0.024 / 0.1 /
# 0.085 (of the fp32 state).  Most of it is fp16 rounding of activations that goes the other way.
_TOLERANCE = {4: {"rel": 1.3e-2, "max": 0.065}, 5.2: {"rel": 1.6e-2, "max": 0.1}, 6: {"rel": 2.6e-2, "max": 0.4},
              7: {"rel": 2.7e-2, "max": 0.35}}


def tolerance(case):
    if case["kind"] == "sample":
        return {"rel": 1e-5, "differ": 0.0}
    if case["kind"] == "mm8":
        # one fp16 rounding of the scaled activation and one of the result: up to 7e-4 / 1.8e-3 from the product in 64 bits
        return {"rel": 2.8e-3, "max": 7e-3}
    return dict(_TOLERANCE[case["version"]])
