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
import torch

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


class _Weights:
    """The random weights of a "synthetic:" model (counter-based: splitmix64, Box-Muller), in the order in which the
    model draws them."""

    def __init__(self, case):
        self.seed, self.drawn, self.quant = 1236 + len(case["weights"]), 0, case["weights"] == "int8"

    @staticmethod
    def _signed(x):
        x &= (1 << 64) - 1
        return x - (1 << 64) if x >> 63 else x

    @classmethod
    def _splitmix(cls, x):
        x = x + cls._signed(0x9E3779B97F4A7C15)
        x = (x ^ ((x >> 30) & ((1 << 34) - 1))) * cls._signed(0xBF58476D1CE4E5B9)
        x = (x ^ ((x >> 27) & ((1 << 37) - 1))) * cls._signed(0x94D049BB133111EB)
        return x ^ ((x >> 31) & ((1 << 33) - 1))

    @classmethod
    def _unit(cls, key, i):
        return (((cls._splitmix(i + key) >> 40) & 0xFFFFFF) + 1).float() * (1.0 / 16777216.0)

    @classmethod
    def _normal(cls, key, i):
        u1, u2 = cls._unit(key, 2 * i), cls._unit(key, 2 * i + 1)
        log = torch.log(u1.double()).float()
        return torch.sqrt(-2.0 * log) * torch.cos((6.2831855 * u2).double()).float()

    def _key(self):
        self.drawn += 1
        x = torch.tensor(self._signed(self.seed * 0x100000001B3 + self.drawn))
        return int(self._splitmix(x))

    def uniform(self, n, lo, hi, half=True):
        v = lo + (hi - lo) * self._unit(self._key(), torch.arange(n, device="cuda"))
        return (v.half() if half else v).double()

    def matrix(self, k, n):
        key, w = self._key(), torch.empty(k, n, device="cuda", dtype=torch.float64)
        rows = max(1, (1 << 25) // n)
        for lo in range(0, k, rows):
            at = torch.arange(lo * n, min(k, lo + rows) * n, device="cuda")
            w[lo:lo + rows] = (0.02 * self._normal(key, at)).half().double().view(-1, n)
        return self._coded(w.float()) if self.quant else w

    @staticmethod
    def _coded(w):
        """What a matrix is in uint8 codes with row and column offsets and ranges in binary16."""
        mx = w.min(0).values.half().float()
        w = w - mx
        my = w.min(1).values.half().float()
        w = w - my[:, None]
        rx = w.max(0).values.clamp(min=1e-4).half().float()
        w = w / rx
        ry = w.max(1).values.clamp(min=1e-4).half().float()
        q = torch.round(w / ry[:, None] * 255.0).clamp(0, 255).double()
        return q * (rx.double() / 255.0) * ry.double()[:, None] + mx.double() + my.double()[:, None]

    def rows(self, ids, c):
        key, at = self._key(), torch.as_tensor(ids, device="cuda", dtype=torch.int64)[:, None] * c
        v = (0.02 * self._normal(key, at + torch.arange(c, device="cuda"))).double()
        return _norm(v).half().double()


def _norm(x):
    return (x - x.mean(-1, keepdim=True)) / torch.sqrt(x.var(-1, unbiased=False, keepdim=True) + 1e-5)


def _running(x, decay):
    """y[t] = decay y[t-1] + x[t], along the first axis."""
    d, n = decay, 1
    while n < len(x):
        x = torch.cat([x[:n], x[n:] + d * x[:-n]])
        d, n = d * d, 2 * n
    return x


def _attention4(w, c, mixed):
    mk, mv, mr = (w.uniform(c, 0, 1) for _ in range(3))
    decay, first = torch.exp(-torch.exp(w.uniform(c, -5, 1, False))), w.uniform(c, -1, 1, False)
    k, v, r = mixed(mk) @ w.matrix(c, c), mixed(mv) @ w.matrix(c, c), torch.sigmoid(mixed(mr) @ w.matrix(c, c))
    e = torch.exp(k)
    num, den = _running(e * v, decay), _running(e, decay)
    now = torch.exp(first + k)
    before = [torch.cat([torch.zeros_like(s[:1]), s[:-1]]) for s in (num, den)]
    return (r * (before[0] + now * v) / (before[1] + now)) @ w.matrix(c, c)


def _attention5(w, c, heads, mixed):
    s = c // heads
    mk, mv, mr, mg = (w.uniform(c, 0, 1) for _ in range(4))
    decay, first = torch.exp(-torch.exp(w.uniform(c, -6, 0, False))), w.uniform(c, -1, 1, False)
    k, v, r, g = (mixed(m) @ w.matrix(c, c) for m in (mk, mv, mr, mg))
    decay, first = decay.view(heads, s, 1), first.view(heads, s, 1)
    state, out = torch.zeros(heads, s, s, device="cuda", dtype=torch.float64), []
    for kt, vt, rt in zip(k.view(-1, heads, s, 1), v.view(-1, heads, 1, s), r.view(-1, heads, 1, s)):
        kv = kt * vt
        out.append(rt @ (state + first * kv))
        state = state * decay + kv
    out = _norm(torch.stack(out).view(-1, heads, s)).view(-1, c)
    return (out * torch.nn.functional.silu(g)) @ w.matrix(c, c)


@torch.no_grad()
def exact(case, seed):
    """The logits in 64 bits, from the weights as the model holds them (binary16, or uint8 codes with their scales)."""
    rng = np.random.default_rng(seed)
    prompt = rng.integers(0, case["vocab"], case["prompt"])
    steps = rng.integers(0, case["vocab"], case["steps"])
    past = rng.integers(0, case["vocab"], 0 if case["fresh"] else 16)
    ids = np.concatenate([past, prompt, steps])
    c, f, w = case["c"], case["f"], _Weights(case)
    table = _Weights(case)
    table.drawn = case["layers"] * (16 if case["heads"] else 14) + 1  # the embedding comes after the layers and the head
    x = table.rows(ids, c)

    for layer in range(case["layers"]):
        def mixed(m):
            return xx * m + torch.cat([torch.zeros_like(xx[:1]), xx[:-1]]) * (1 - m)
        xx = _norm(x)
        x = x + (_attention5(w, c, case["heads"], mixed) if case["heads"] else _attention4(w, c, mixed))
        xx = _norm(x)
        mk, mr = w.uniform(c, 0, 1), w.uniform(c, 0, 1)
        k = torch.relu(mixed(mk) @ w.matrix(c, f)) ** 2
        v = k @ w.matrix(f, c)
        x = x + v * torch.sigmoid(mixed(mr) @ w.matrix(c, c))
        if (layer + 1) % 6 == 0:
            x = x / 2
    if not case["score"]:
        x = x[(len(past) if len(prompt) == 0 else len(past) + len(prompt) - 1):]
    logits = (_norm(x) @ w.matrix(c, case["vocab"])).cpu().numpy()
    return logits if case["score"] else list(logits)
