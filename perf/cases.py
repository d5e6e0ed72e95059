"""Workloads of the quantized-linear backend, as a program that uses it issues them.

Three paths, all through the public entry points (``GEMV``, ``GEMVGroup``, ``TiedEmbedding`` and the
table ops of ``coffin_amd.backend``):

* ``step``    the projection side of a model step: embedding lookup, per layer norm -> q/k/v ->
              o -> add + norm -> gate/up -> SiLU product -> down, final norm, ``lm_head``.  What lies
              between q/k/v and o (attention) is not this framework's, so its output is an input here.
              ``entry`` says in which of the four roles the projections are called: ``decode`` (one
              sequence), ``static`` (a batch of sequences), ``verify`` (a speculative window) or
              ``prefill`` (a chunk of a prompt, whose last row alone goes through ``lm_head``).
              ``captured``: the step is replayed from a HIP graph, as a serving loop replays it.
* ``mlp``     norm -> gate/up -> SiLU product -> down alone.
* ``linear``  one projection.
* ``kv``      the per-row int8 quantiser on the key and value rows that a chunk adds to its cache.

Weights are N(0, 0.02) through the package's own encoders, activations N(0, 1) in bf16, 1 % of them
20 times larger in prefill.
"""

from __future__ import annotations

import math

import torch

from coffin_amd import backend
from coffin_amd.embed import TiedEmbedding
from coffin_amd.gemv import GEMV, GEMVGroup
from coffin_amd.weights import QWeight, W4A8Weight

#: The 4B-shaped model of the package's benchmark and tests.
MODEL = {"hidden": 2560, "q": 4096, "kv": 1024, "inter": 9728, "vocab": 151936}


def _step(name, weights, entry, rows, layers, captured=False, family="", group=128, **sizes):
    return {"name": name, "path": "step", "weights": weights, "entry": entry, "rows": rows, "layers": layers,
            "captured": captured, "family": family, "group": group, **{**MODEL, **sizes}}


def listed() -> list:
    return [
        # The smallest call a decode loop makes: the unfused key projection of one token.
        {"name": "k projection, 1 row", "path": "linear", "weights": "int8", "entry": "decode", "rows": 1,
         "k": 2560, "n": 1024, "family": "", "group": 128},
        # One token of one sequence, int8 and int4 weights, called eagerly (development, first tokens,
        # anything that cannot be captured).
        _step("token, int8", "int8", "decode", 1, 4),
        _step("token, int4", "int4", "decode", 1, 4),
        # The same token as serving runs it.
        _step("token, int8, captured", "int8", "decode", 1, 8, captured=True),
        # Static batches: a few sequences on int8 weights, sixteen on int4.
        _step("batch of 4, int8", "int8", "static", 4, 2),
        _step("batch of 16, int4", "int4", "static", 16, 2),
        # Prompts: a short one, a chat-sized one of no round length, the engine's chunk (2048), and a
        # long prompt in one piece.
        _step("prompt of 100, int4", "int4", "prefill", 100, 2),
        _step("prompt of 500, int8", "int8", "prefill", 500, 2),
        _step("prompt of 2048, int8", "int8", "prefill", 2048, 2),
        _step("prompt of 8192, int8", "int8", "prefill", 8192, 2),
        # The MLP of a larger dense model on int4 weights, 1024 rows.
        {"name": "large mlp of 1024, int4", "path": "mlp", "weights": "int4", "entry": "prefill", "rows": 1024,
         "hidden": 5120, "inter": 25600, "family": "", "group": 128},
        # Keys and values of a 2048-token chunk (8 heads of 128) on their way into an int8 cache.
        {"name": "cache rows of 2048 tokens", "path": "kv", "rows": 2048 * 8, "width": 128},
    ]


# ------------------------------------------------------------------------------ drawn cases

def _log(rng, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _width(rng, lo: int, hi: int) -> int:
    """A model width: whole 128s mostly, whole 64s otherwise."""
    unit = 128 if rng.random() < 0.7 else 64
    return max(1, round(_log(rng, lo, hi) / unit)) * unit


def _rows(rng, entry: str) -> int:
    return {"decode": lambda: 1, "static": lambda: rng.randint(2, 16), "verify": lambda: rng.randint(2, 9),
            "prefill": lambda: round(_log(rng, 9, 8192))}[entry]()


def _seconds(case) -> float:
    """A coarse bound on what a case takes, to keep drawn ones below the largest listed one."""
    w = work(case)
    return w["bytes"] / 2e12 + w["flops"] / 5e14


def draw(rng) -> dict:
    limit = max(_seconds(c) for c in listed())
    while True:
        path = rng.choices(("linear", "step", "mlp", "kv"), (0.35, 0.35, 0.15, 0.15))[0]
        if path == "kv":
            case = {"path": "kv", "rows": round(_log(rng, 2, 65536)), "width": rng.choice((64, 96, 128, 192, 256, 512, 576))}
        else:
            entry = rng.choices(("decode", "static", "verify", "prefill"), (0.25, 0.15, 0.15, 0.45))[0]
            weights = rng.choice(("int8", "int4"))
            case = {"path": path, "weights": weights, "entry": entry, "rows": _rows(rng, entry),
                    "family": "mfma" if weights == "int8" and entry == "static" and rng.random() < 0.3 else "",
                    "group": rng.choices((128, 64, 256), (0.8, 0.1, 0.1))[0] if weights == "int4" else 128}
            if path == "linear":
                case["k"] = _width(rng, 512, 25600)
                case["n"] = round(_log(rng, 256, 32768))
                if weights == "int4" and rng.random() < 0.1:
                    case["k"] += rng.randint(1, 63)        # rows that are not whole groups
            else:
                case["hidden"] = _width(rng, 512, 5120)
                case["inter"] = _width(rng, 2 * case["hidden"], 5 * case["hidden"])
            if path == "step":
                heads = rng.randint(4, 40)
                case.update(q=128 * heads, kv=128 * rng.randint(1, min(heads, 16)), vocab=round(_log(rng, 8000, 160000)),
                            layers=rng.randint(1, 3), captured=entry != "prefill" and rng.random() < 0.3)
        if _seconds(case) <= limit:
            return case


# ------------------------------------------------------------------------------ inputs

def _dense(n: int, k: int, gen: torch.Generator) -> torch.Tensor:
    return torch.randn((n, k), generator=gen, device="cuda") * 0.02


def _weight(case, n: int, k: int, gen: torch.Generator):
    if case["weights"] == "int8":
        w = QWeight.quantize(_dense(n, k, gen))
        w.batch_family = case["family"] or None
        return w
    return W4A8Weight.quantize(_dense(n, k, gen), case["group"])


def _group(case, sizes: list, k: int, gen: torch.Generator) -> GEMVGroup:
    group = GEMVGroup([_weight(case, n, k, gen) for n in sizes])
    if case["weights"] == "int8":
        group.g.w.batch_family = case["family"] or None
    return group


def _gain(n: int, gen: torch.Generator) -> torch.Tensor:
    return (1 + 0.1 * torch.randn(n, generator=gen, device="cuda")).to(torch.bfloat16)


def _activations(case, rows: int, k: int, gen: torch.Generator) -> torch.Tensor:
    x = torch.randn((rows, k), generator=gen, device="cuda")
    if case["path"] != "kv" and case["entry"] == "prefill":
        x = torch.where(torch.rand((rows, k), generator=gen, device="cuda") < 0.01, x * 20.0, x)
    return x.to(torch.bfloat16)


def _call(entry: str):
    """How a projection (``GEMV`` or ``GEMVGroup``) is called in this role."""
    return {"decode": lambda p, x: p(x), "static": lambda p, x: p.linear_m(x),
            "verify": lambda p, x: p.linear_m_verify(x), "prefill": lambda p, x: p.prefill(x)}[entry]


class _Linear:
    def __init__(self, case, gen) -> None:
        self.proj, self.call = GEMV(_weight(case, case["n"], case["k"], gen)), _call(case["entry"])
        self.x = _activations(case, case["rows"], case["k"], gen)

    def __call__(self):
        return self.call(self.proj, self.x)


class _Mlp:
    def __init__(self, case, gen) -> None:
        rows, hidden, inter = case["rows"], case["hidden"], case["inter"]
        self.call = _call(case["entry"])
        self.gate_up, self.down = _group(case, [inter, inter], hidden, gen), GEMV(_weight(case, hidden, inter, gen))
        self.gain, self.x = _gain(hidden, gen), _activations(case, rows, hidden, gen)
        self.act = torch.empty((rows, inter), dtype=torch.bfloat16, device="cuda")

    def __call__(self):
        gate, up = self.call(self.gate_up, backend.rms_norm(self.x, self.gain))
        return self.call(self.down, backend.silu_mul(gate, up, self.act))


class _Step:
    def __init__(self, case, gen) -> None:
        rows, hidden, inter = case["rows"], case["hidden"], case["inter"]
        self.call, self.last_row = _call(case["entry"]), case["entry"] == "prefill"
        self.embed = TiedEmbedding(_weight(case, case["vocab"], hidden, gen))
        self.ids = torch.randint(0, case["vocab"], (rows,), generator=gen, device="cuda")
        self.layers = [(_group(case, [case["q"], case["kv"], case["kv"]], hidden, gen),
                        GEMV(_weight(case, hidden, case["q"], gen)),
                        _group(case, [inter, inter], hidden, gen),
                        GEMV(_weight(case, hidden, inter, gen)),
                        _gain(hidden, gen),
                        _activations(case, rows, case["q"], gen)) for _ in range(case["layers"])]
        self.gains = [_gain(hidden, gen) for _ in range(case["layers"] + 1)]
        # workspaces a program keeps: the normalised rows and the SiLU product
        self.h = torch.empty((rows, hidden), dtype=torch.bfloat16, device="cuda")
        self.act = torch.empty((rows, inter), dtype=torch.bfloat16, device="cuda")
        self.graph = None
        if case["captured"]:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                self()
            torch.cuda.current_stream().wait_stream(side)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                self.out = self()
            self.graph = graph

    def __call__(self):
        if self.graph is not None:
            self.graph.replay()
            return self.out
        call, seen = self.call, []
        x = self.embed.lookup(self.ids)
        h = backend.rms_norm(x, self.gains[0])
        for (qkv, o, gate_up, down, gain, attn), after in zip(self.layers, self.gains[1:]):
            seen += call(qkv, h)
            h = backend.add_rms_norm(x, call(o, attn), gain, self.h)
            gate, up = call(gate_up, h)
            y = call(down, backend.silu_mul(gate, up, self.act))
            h = backend.add_rms_norm(x, y, after, self.h)
        logits = self.embed(h[-1]) if self.last_row else call(self.embed.gemv, h)
        return [*seen, x, logits]


class _Kv:
    def __init__(self, case, gen) -> None:
        rows, width = case["rows"], case["width"]
        self.parts = [(_activations(case, rows, width, gen),
                       torch.empty((rows, width), dtype=torch.int8, device="cuda"),
                       torch.empty(rows, dtype=torch.float32, device="cuda")) for _ in ("keys", "values")]

    def __call__(self):
        for x, q, s in self.parts:
            backend.kv_quant(x, q, s)
        return [t for _, q, s in self.parts for t in (q, s)]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return {"linear": _Linear, "mlp": _Mlp, "step": _Step, "kv": _Kv}[case["path"]](case, gen)


def run(state):
    return state()


# ------------------------------------------------------------------------------ costs and tolerances

def _weight_bytes(case, n: int, k: int) -> float:
    return n * k + 4 * n if case["weights"] == "int8" else n * k / 2 + 4 * n * math.ceil(k / case["group"])


def work(case) -> dict:
    """Stored weights, inputs and outputs once; multiply-adds of the projections as two operations."""
    path, rows = case["path"], case["rows"]
    if path == "kv":
        elements = 2 * rows * case["width"]
        return {"bytes": 3 * elements + 8 * rows, "flops": 3 * elements}
    if path == "linear":
        n, k = case["n"], case["k"]
        return {"bytes": _weight_bytes(case, n, k) + 2 * rows * (n + k), "flops": 2 * rows * n * k}
    hidden, inter = case["hidden"], case["inter"]
    shapes = [(2 * inter, hidden), (hidden, inter)]
    if path == "mlp":
        return {"bytes": sum(_weight_bytes(case, n, k) for n, k in shapes) + 2 * hidden + 4 * rows * hidden,
                "flops": sum(2 * rows * n * k for n, k in shapes)}
    qkv = case["q"] + 2 * case["kv"]
    shapes += [(qkv, hidden), (hidden, case["q"])]
    heads = 1 if case["entry"] == "prefill" else rows
    layer = sum(_weight_bytes(case, n, k) for n, k in shapes) + 2 * rows * (case["q"] + qkv) + 4 * hidden
    looked_up = rows * _weight_bytes(case, 1, hidden) + 8 * rows
    head = _weight_bytes(case, case["vocab"], hidden) + 2 * heads * case["vocab"]
    return {"bytes": case["layers"] * layer + looked_up + head + 2 * rows * hidden + 2 * hidden,
            "flops": case["layers"] * sum(2 * rows * n * k for n, k in shapes) + 2 * heads * case["vocab"] * hidden}


def tolerance(case):
    """The quantiser's results are specified to the bit; everything else is bf16 with fp32 sums."""
    return "exact" if case["path"] == "kv" else {"rel": 1e-2}
