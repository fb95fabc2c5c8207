"""The work that programs have this backend do, as measured cases.

A case is one model shape, one weight type and one request to it, run through `Model` as a program does: a prompt
(`Model.run` on several ids), then tokens one at a time (`Model.run` on one id) -- the loop of a program that picks each
token itself from the logits -- or the logits of every position of a text (`Model.run_full`).  The tokens that are fed
come with the case, so that the logits of two builds can be compared value by value; whether a pass left the right
recurrent state behind shows in the logits of the tokens that follow it.

The widths are those of the RWKV models that the tests and the benchmark run (169M, 1.5B, 3B, 7B and 14B); the widest
ones and RWKV-5.2 with fewer layers than the models have, every layer being the same work again.  (RWKV-5.2 with random
weights and all 32 layers amplifies the rounding of any one sum into the tenths of a logit; with 12 it does not.)
"""
import importlib
import math

import numpy as np

fr = importlib.import_module("faster-rwkv_amd")

# name: RWKV version, layers, width, ffn width, vocabulary, heads
SHAPES = {
    "v4-169m": ("4", 12, 768, 3072, 50277, 0),
    "v4-1b5": ("4", 24, 2048, 8192, 65536, 0),
    "v5-3b": ("5.2", 12, 2560, 8960, 65536, 40),
    "v5-7b": ("5.2", 2, 4096, 14336, 65536, 64),
    "v4-14b": ("4", 2, 5120, 20480, 65536, 0),
}


def _case(name, shape, weights, prompt, steps, fresh, score=False):
    v, layers, c, f, vocab, heads = SHAPES[shape]
    return {"name": name, "version": v, "layers": layers, "c": c, "f": f, "vocab": vocab, "heads": heads,
            "weights": weights, "prompt": prompt, "steps": steps, "fresh": fresh, "score": score}


def listed():
    return [
        # Generation token by token inside a conversation: the small model, where a token is launches and latency ...
        _case("decode-169m-fp16", "v4-169m", "fp16", 0, 8, False),
        # ... the model of the headline benchmark in both weight types ...
        _case("decode-1b5-fp16", "v4-1b5", "fp16", 0, 8, False),
        _case("decode-1b5-int8", "v4-1b5", "int8", 0, 8, False),
        # ... a model with the matrix-valued state ...
        _case("decode-v5-3b-int8", "v5-3b", "int8", 0, 8, False),
        # ... and the widest one.
        _case("decode-14b-fp16", "v4-14b", "fp16", 0, 8, False),
        # A short turn of a conversation: a line of text, read on top of the state so far, and the answer's beginning.
        _case("turn-13-1b5-int8", "v4-1b5", "int8", 13, 2, False),
        # New requests, from an empty state: a question, a page, a long document ...
        _case("prompt-77-1b5-fp16", "v4-1b5", "fp16", 77, 1, True),
        _case("prompt-1024-1b5-fp16", "v4-1b5", "fp16", 1024, 1, True),
        _case("prompt-4099-1b5-fp16", "v4-1b5", "fp16", 4099, 1, True),
        # ... and the same with the matrix-valued state, in both weight types.
        _case("prompt-512-v5-3b-int8", "v5-3b", "int8", 512, 1, True),
        _case("prompt-300-v5-7b-fp16", "v5-7b", "fp16", 300, 1, True),
        # The likelihood of a text under the small model: the logits of every position.
        _case("score-256-169m-fp16", "v4-169m", "fp16", 256, 0, True, score=True),
    ]


def draw(rng):
    """A model of a width and depth inside the listed ranges, and a request to it."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    version = rng.choice(["4", "5.2"])
    c = 128 * log_int(768 // 128, 5120 // 128)
    f = 4 * c if version == "4" else 7 * c // 2
    layers = min(12, max(2, int(2.5e8 / (6 * c * c + 2 * c * f))))
    vocab = rng.choice([8192, 50277, 65536])
    case = {"version": version, "layers": layers, "c": c, "f": f, "vocab": vocab,
            "heads": c // 64 if version == "5.2" else 0, "weights": rng.choice(["fp16", "int8"]), "score": False}
    kind = rng.choice(["decode", "turn", "prompt", "prompt", "score"])
    if kind == "decode":
        case.update(prompt=0, steps=rng.randint(4, 12), fresh=False)
    elif kind == "turn":
        case.update(prompt=log_int(4, 128), steps=rng.randint(1, 4), fresh=False)
    elif kind == "prompt":
        case.update(prompt=log_int(16, 4096), steps=1, fresh=True)
    else:
        case.update(prompt=log_int(16, 256), steps=0, fresh=True, score=True)
    return case


_models = {}


def _model(case):
    """The loaded model, as a serving program keeps it: one per shape and weight type."""
    key = tuple(case[k] for k in ("version", "layers", "c", "f", "vocab", "heads", "weights"))
    if key not in _models:
        spec = "synthetic:v=%s,L=%d,C=%d,F=%d,V=%d,seed=%d" % (key[:5] + (1236 + len(case["weights"]),))
        if case["heads"]:
            spec += ",H=%d" % case["heads"]
        _models[key] = fr.Model(spec, "hip " + case["weights"])
    return _models[key]


def prepare(case, seed):
    model = _model(case)
    rng = np.random.default_rng(seed)
    state = {"model": model, "fresh": case["fresh"], "score": case["score"],
             "prompt": rng.integers(0, case["vocab"], case["prompt"]).astype(np.int32),
             "steps": [int(t) for t in rng.integers(0, case["vocab"], case["steps"])]}
    if not case["fresh"]:  # the conversation so far
        model.reset()
        model.run(rng.integers(0, case["vocab"], 16).astype(np.int32))
    return state


def run(state):
    model = state["model"]
    if state["fresh"]:
        model.reset()
    if state["score"]:
        return model.run_full(state["prompt"])
    logits = [model.run(state["prompt"])] if len(state["prompt"]) else []
    logits += [model.run(t) for t in state["steps"]]
    return logits


def work(case):
    """Every matrix weight once per pass over it (a prompt is one pass, a token another), uint8 weights with their
    scales, the recurrent state in and out, embedding rows in and logits out."""
    c, f, v, layers = case["c"], case["f"], case["vocab"], case["layers"]
    v5 = case["version"] != "4"
    mats = [(c, c)] * (6 if v5 else 5) + [(c, f), (f, c)]
    size = (lambda k, n: 2 * k * n) if case["weights"] == "fp16" else (lambda k, n: k * n + 4 * (k + n))
    body = layers * sum(size(k, n) for k, n in mats)
    head = size(c, v)
    state = layers * 2 * (2 * 2 * c + (4 * 64 * c if v5 else 3 * 4 * c))
    # per token: the products; the scan of the state (RWKV-5: decay, rank-one update and read-out of [64, 64] per head)
    token = layers * (2.0 * sum(k * n for k, n in mats) + (6.0 * 64 * c if v5 else 20.0 * c))
    passes = ([case["prompt"]] if case["prompt"] else []) + [1] * case["steps"]
    total = {"bytes": 0.0, "flops": 0.0}
    for t in passes:
        rows = t if case["score"] else 1
        total["bytes"] += body + head + state + 2.0 * c * t + 4.0 * v * rows
        total["flops"] += token * t + 2.0 * c * v * rows
    return total


def tolerance(case):
    """Activations are binary16, rounded after every operation, so two valid orders of the products' sums drift apart.
    Measured between prompts as one pass and as one-token steps: RWKV-4 up to 3.6e-3 of the logits' norm, the largest
    difference 1.6e-2 of their rms; RWKV-5.2 5.4e-3 and 2.2e-2.  Four times that."""
    return {"rel": 0.015, "max": 0.065} if case["version"] == "4" else {"rel": 0.022, "max": 0.09}
