"""What a user of the framework has it do, as timed cases over its public entry points.

Three kinds of case:

- ``step``: one ``Dion.step()`` over the parameters of a model (or of the part of one that a
  training process holds): matrices by their shapes per layer, vectors and tables on AdamW,
  with or without an EMA of the weights on the GPU. Gradients are in ``.grad``, the state is
  that of a run under way (non-zero momentum, row variances, AdamW moments, shadows).
- ``orthogonalize``: ``newton_schulz_fn(kind)(batch, eps)``, the operator that a program with an
  optimizer of its own calls on a batch of updates.
- ``ema``: ``foreach_ema_update_`` of a list of weights, as a program that keeps its own average
  calls it.

``exact`` restates each in float64 with plain torch.
"""

from __future__ import annotations

import math

import torch

import dionw_amd
from dionw_amd.ema._update import foreach_ema_update_
from dionw_amd.newton_schulz import NewtonSchulz, newton_schulz_fn

LR, MOMENTUM, BETA2, BETAS, EPS = 3e-4, 0.95, 0.95, (0.9, 0.95), 1e-8
EMA_DECAY = 0.9999
ADAMW_STEPS = 100.0  # steps that the AdamW state has behind it
NS_EPS = 1e-8
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}


def _step(name: str, matrices: str, layers: int, **options) -> dict:
    """A step over ``layers`` layers. ``matrices``: ROWSxCOLS[*count][/heads] per layer,
    ``vectors``: LENGTH[*count] per layer, ``tables``: ROWSxCOLS[*count] once."""
    case = {"name": name, "kind": "step", "matrices": matrices, "layers": layers, "vectors": "",
            "tables": "", "fraction": 1.0, "update": "dion3", "iteration": "gram", "decay": 0.05,
            "ema": False, "heavy_tails": False}
    return {**case, **options}


def listed() -> list[dict]:
    return [
        # One square weight, every row: the least work a step can have (latency).
        _step("step-1-weight-1024", "1024x1024", 1),
        # A small model of odd sizes, rows selected, an EMA: side 200 is no multiple of 32,
        # the 4-head projection splits into 50-row blocks.
        _step("step-odd-200", "600x200,200x200/4,777x200,200x777", 6, vectors="200*4,777",
              tables="5003x200", fraction=0.3, ema=True),
        # The GPT-2-small-shaped parameter set, all of it.
        _step("step-gpt2-small", "2304x768,768x768,3072x768,768x3072", 12,
              vectors="2304,768*6,3072", tables="50257x768,1024x768"),
        # Llama-3-8B-shaped layers with a quarter of the rows selected: four of the 32 and one
        # of the two vocabulary tables, as a process that holds an eighth of the model steps.
        _step("step-llama-4-layers",
              "4096x4096,1024x4096,1024x4096,4096x4096,14336x4096,14336x4096,4096x14336", 4,
              vectors="4096*2", tables="128256x4096", fraction=0.25),
        # An MoE expert stack: 64 experts, heavy-tailed gradients, rows selected, GPU EMA.
        _step("step-moe-64-ema", "1408x2048,1408x2048,2048x1408", 64, fraction=0.25, ema=True,
              heavy_tails=True),
        # The same stack under plain Muon: bf16 quintic, Nesterov momentum, every row.
        _step("step-moe-64-muon", "1408x2048,1408x2048,2048x1408", 64, update="muon",
              iteration="keller_triton", heavy_tails=True),
        # A batch of wide updates in bf16.
        _orthogonalize("gram-16x1024x4096", "gram", 16, 1024, 4096, "bfloat16"),
        # Tall updates in float32 (the transposed orientation), a side that tiles leave ragged.
        _orthogonalize("gram-28x1152x576", "gram", 28, 1152, 576, "float32"),
        # One large update alone, as a process that owns one layer's matrix has it.
        _orthogonalize("gram-1x3584x4096", "gram", 1, 3584, 4096, "float32"),
        # The longest rows, through the bf16 Polar Express quintic.
        _orthogonalize("polar-16x1024x8192", "polar_express_triton", 16, 1024, 8192, "bfloat16"),
        # A few updates of odd sides in float16.
        _orthogonalize("keller-3x500x1301", "keller", 3, 500, 1301, "float16"),
        # A program's own weight average over a table, some matrices and vectors.
        {"name": "ema-46M", "kind": "ema", "shapes": "50257x768,768x768*12,768*25"},
    ]


def _orthogonalize(name: str, iteration: str, blocks: int, rows: int, cols: int,
                   dtype: str) -> dict:
    return {"name": name, "kind": "orthogonalize", "iteration": iteration, "blocks": blocks,
            "rows": rows, "cols": cols, "dtype": dtype}


def _log_int(rng, low: float, high: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _side(rng, low: float, high: float) -> int:
    """A size, spread over its logarithm: any integer, or a multiple of 8 or 64."""
    n, unit = _log_int(rng, low, high), rng.choice([1, 8, 64, 64])
    return max(unit, n // unit * unit)


def draw(rng) -> dict:
    kind = rng.choices(["step", "experts", "orthogonalize", "ema"], [4, 2, 5, 1])[0]
    if kind == "orthogonalize":
        iteration = rng.choice(["gram", "gram", "polar_express_triton", "polar_express", "keller",
                                "keller_triton"])
        short = _side(rng, 64, 3584)
        long = short if rng.random() < 0.15 else int(short * rng.choice([1.25, 2, 3, 4, 8]))
        long = max(short, min(long, 16384))
        each = _flops(iteration, short, long)
        blocks = _log_int(rng, 1, max(1.0, min(64.0, 4e12 / each)))
        rows, cols = (long, short) if rng.random() < 0.4 else (short, long)
        case = _orthogonalize("", iteration, blocks, rows, cols,
                              rng.choice(["float32", "bfloat16", "float16"]))
    elif kind == "ema":
        width = _side(rng, 64, 4096)
        case = {"kind": "ema", "shapes": "%dx%d,%dx%d*%d,%d*%d" % (
            _log_int(rng, 100, 40000), width, _log_int(rng, 64, 2048), width, rng.randint(1, 12),
            width, rng.randint(1, 60))}
    else:
        width = _side(rng, 64, 4096 if kind == "step" else 2048)
        inner = int(width * rng.choice([2.6875, 3, 3.5, 4] if kind == "step" else [0.5, 0.6875, 1.5]))
        if kind == "step":
            heads = rng.choice(["", "", "/4" if width % 4 == 0 else ""])
            matrices = "%dx%d%s,%dx%d,%dx%d,%dx%d" % (3 * width, width, heads, width, width,
                                                      inner, width, width, inner)
            vectors, most = "%d*4,%d" % (width, inner), 24
        else:
            matrices = "%dx%d*2,%dx%d" % (inner, width, width, inner)
            vectors, most = "", 64
        fraction = rng.choice([1.0, 0.5, 0.25, 0.25])
        update = "muon" if fraction == 1.0 and rng.random() < 0.5 else "dion3"
        iteration = "keller_triton" if update == "muon" else rng.choice(
            ["gram", "gram", "polar_express_triton"])
        case = _step("", matrices, 1, vectors=vectors, fraction=fraction, update=update,
                     iteration=iteration, decay=rng.choice([0.05, 0.05, 0.0]),
                     ema=rng.random() < 0.3, heavy_tails=rng.random() < 0.3)
        one = work(case)
        fit = min(most, 5e8 * 20 / one["bytes"], 5e12 / one["flops"])
        case["layers"] = _log_int(rng, 1, max(1.0, fit))
        if kind == "step":
            case["tables"] = "%dx%d" % (_log_int(rng, 256, 32000), width)
    case.pop("name", None)
    return case


# ---- shapes and work ---------------------------------------------------------------

def _shapes(text: str) -> list[tuple[tuple[int, ...], int, int | None]]:
    """[(shape, count, heads)] of a list of ROWSxCOLS[*count][/heads]."""
    out = []
    for item in filter(None, text.split(",")):
        item, _, heads = item.partition("/")
        item, _, count = item.partition("*")
        out.append((tuple(int(n) for n in item.split("x")), int(count or 1),
                    int(heads) if heads else None))
    return out


def _selected(rows: int, fraction: float) -> int:
    return min(rows, math.ceil(fraction * rows))


def _flops(iteration: str, rows: int, cols: int) -> float:
    """The iteration's products on one block, of the symmetric ones the upper half only."""
    r, c = float(min(rows, cols)), float(max(rows, cols))
    if iteration == "gram" and c > r:
        return 6 * r * r * c + 14 * r ** 3
    return 15 * r * r * c + 5 * r ** 3


def work(case: dict) -> dict:
    if case["kind"] == "orthogonalize":
        n, rows, cols = case["blocks"], case["rows"], case["cols"]
        size = 4 if case["dtype"] == "float32" else 2
        return {"bytes": n * rows * cols * (size + 2),
                "flops": n * _flops(case["iteration"], rows, cols)}
    if case["kind"] == "ema":
        n = sum(math.prod(shape) * count for shape, count, _ in _shapes(case["shapes"]))
        return {"bytes": 12 * n, "flops": 3 * n}
    ema = 8 if case["ema"] else 0  # shadow read and written
    size = flops = 0.0
    for (rows, cols), count, heads in _shapes(case["matrices"]):
        heads = heads or 1
        k = _selected(rows // heads, case["fraction"])
        n = count * case["layers"]
        # gradient read, momentum read and written, weight read and written (where no
        # decay applies, on the selected rows only)
        written = rows if case["decay"] or ema else k * heads
        size += n * cols * (12 * rows + 8 * written + ema * rows)
        flops += n * heads * _flops(case["iteration"], k, cols)
    adamw = sum(shape[0] * count for shape, count, _ in _shapes(case["vectors"])) * case["layers"]
    adamw += sum(math.prod(shape) * count for shape, count, _ in _shapes(case["tables"]))
    return {"bytes": size + (28 + ema) * adamw, "flops": flops + 12 * adamw}


def tolerance(case: dict) -> dict:
    if case["kind"] == "ema":
        return {"rel": 1e-6}
    # The iterations against their float64 polynomials: 0.002 to 0.003 measured for the float16
    # Gram iteration, 0.01 to 0.02 for the bf16 quintics.
    gram = case["iteration"] == "gram"
    if case["kind"] == "orthogonalize":
        return {"rel": 0.01 if gram else 0.03}
    # Of a step's outputs the row variances carry most of that error: 1e-5 to 3e-4 measured
    # with Gram, the weights 6e-6 to 4e-5.
    return {"rel": 0.001 if gram else 0.004}


# ---- inputs --------------------------------------------------------------------------

class _Stack:
    """``count`` equally shaped float32 tensors, each from an aligned place of its own, which
    one strided tensor (``whole``) shows together."""

    def __init__(self, shape: tuple[int, ...], count: int) -> None:
        numel = math.prod(shape)
        pitch = (numel + 127) // 128 * 128
        self.shape, self.count = shape, count
        store = torch.zeros(count * pitch, device="cuda")
        strides = [1]
        for n in reversed(shape[1:]):
            strides.insert(0, strides[0] * n)
        self.whole = store.as_strided((count, *shape), (pitch, *strides))

    def __getitem__(self, i: int) -> torch.Tensor:
        return self.whole[i]


def _normal(g, shape, scale: float) -> torch.Tensor:
    return torch.empty(shape, device="cuda").normal_(0.0, scale, generator=g)


def _gradient(g, shape, heavy_tails: bool) -> torch.Tensor:
    """1e-3 N(0, 1), or 1e-3 Student-t with 3 degrees of freedom."""
    x = _normal(g, shape, 1e-3)
    if heavy_tails:
        square = torch.zeros(shape, device="cuda")
        for _ in range(3):
            square += _normal(g, shape, 1.0).square_()
        x /= square.mul_(1 / 3).sqrt_().clamp_(min=1e-3)
    return x


def _uniform(g, shape, low: float, high: float) -> torch.Tensor:
    return torch.empty(shape, device="cuda").uniform_(low, high, generator=g)


def _fill(g, case: dict, matrices, adamw) -> None:
    """Weights, gradients and state of a run under way, from the generator alone."""
    heavy = case["heavy_tails"]
    for m in matrices:
        shape = m["w"].whole.shape
        rows, cols = shape[1] // m["heads"], shape[2]
        k = _selected(rows, case["fraction"])
        m["w"].whole.copy_(_normal(g, shape, 0.02))
        m["g"].whole.copy_(_gradient(g, shape, heavy))
        m["m"].copy_(_normal(g, shape, 3e-3))
        m["v"].copy_(_uniform(g, m["v"].shape, 0.8 / max(k, cols), 1.2 / max(k, cols)))
    for a in adamw:
        shape = a["w"].whole.shape
        a["w"].whole.copy_(_normal(g, shape, 0.02))
        a["g"].whole.copy_(_normal(g, shape, 1e-3))
        a["m"].whole.copy_(_normal(g, shape, 3e-4))
        a["v"].whole.copy_(_uniform(g, shape, 5e-7, 2e-6))
    for s in (*matrices, *adamw):
        if "s" in s:
            s["s"].whole.copy_(s["w"].whole + _normal(g, s["w"].whole.shape, 2e-3))


def _lists(case: dict) -> tuple[dict, list]:
    """The step's matrices by (shape, heads) and its AdamW stacks as (shape, count, decayed)."""
    matrices: dict = {}
    for shape, count, heads in _shapes(case["matrices"]):
        key = (shape, heads)
        matrices[key] = matrices.get(key, 0) + count
    matrices = {key: n * case["layers"] for key, n in matrices.items()}
    adamw = [(shape, count, True) for shape, count, _ in _shapes(case["tables"])]
    adamw += [(shape, count * case["layers"], False) for shape, count, _ in _shapes(case["vectors"])]
    return matrices, adamw


def _prepare_step(case: dict, seed: int) -> dict:
    shapes, vectors = _lists(case)
    matrices, adamw = [], []
    groups = []
    for shape, count, decayed in vectors:
        a = {"w": _Stack(shape, count), "g": _Stack(shape, count), "m": _Stack(shape, count),
             "v": _Stack(shape, count), "decay": case["decay"] if decayed else 0.0}
        a["params"] = [torch.nn.Parameter(a["w"][i]) for i in range(count)]
        adamw.append(a)
    for decay in sorted({a["decay"] for a in adamw}):
        groups.append({"params": [p for a in adamw if a["decay"] == decay for p in a["params"]],
                       "dion_route": "adamw", "weight_decay": decay})
    for (shape, heads), count in shapes.items():
        m = {"w": _Stack(shape, count), "g": _Stack(shape, count), "heads": heads or 1}
        m["params"] = [torch.nn.Parameter(m["w"][i]) for i in range(count)]
        matrices.append(m)
    for heads in dict.fromkeys(h for _, h in shapes):
        groups.append({"params": [p for m in matrices if m["heads"] == (heads or 1)
                                  for p in m["params"]],
                       "dion_route": "matrix", "fraction": case["fraction"], "num_heads": heads,
                       "newton_schulz": case["iteration"]})
    opt = dionw_amd.Dion(
        groups, lr=LR, momentum=MOMENTUM, muon_beta2=BETA2, betas=BETAS,
        weight_decay=case["decay"], eps=EPS,
        matrix_update=dionw_amd.MUON_UPDATE if case["update"] == "muon" else dionw_amd.DION3_UPDATE,
        ema=dionw_amd.EMAConfig(decay=EMA_DECAY) if case["ema"] else None)
    for s in (*matrices, *adamw):
        for i, p in enumerate(s["params"]):
            p.grad = s["g"][i]
    if case["ema"]:
        opt.step()  # the first step sets the shadows; its result is written over below
    for a in adamw:
        for i, p in enumerate(a["params"]):
            opt.initialize_state(p)
            opt.state[p].update({"exp_avg": a["m"][i], "exp_avg_sq": a["v"][i]})
            opt.state[p]["adamw_step"].fill_(ADAMW_STEPS)
    for m in matrices:
        opt.initialize_state(m["params"][0])
        # The momenta (and row variances) of equally shaped blocks are one tensor.
        count, shape = m["w"].count, m["w"].shape
        first = opt.state[m["params"][0]]
        m["m"] = first["momentum"].as_strided((count, *shape), (math.prod(shape), shape[1], 1))
        m["v"] = first["variance"].as_strided((count, shape[0]), (shape[0], 1))
    if case["ema"]:
        for s in (*matrices, *adamw):
            s["s"] = _Stack(s["w"].shape, s["w"].count)
            for i, p in enumerate(s["params"]):
                opt.state[p]["ema_shadow"] = s["s"][i]
    _fill(torch.Generator(device="cuda").manual_seed(seed), case, matrices, adamw)
    outputs = {}
    for i, s in enumerate((*matrices, *adamw)):
        for key in "wmvs":
            if key in s:
                outputs["%d%s" % (i, key)] = s[key].whole if isinstance(s[key], _Stack) else s[key]
    return {"opt": opt, "outputs": outputs, "matrices": matrices, "adamw": adamw}


def _updates(case: dict, seed: int) -> torch.Tensor:
    """A batch of updates whose rows differ in size, as gradients' do."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = _normal(g, (case["blocks"], case["rows"], case["cols"]), 1e-3)
    x *= _normal(g, (case["blocks"], case["rows"], 1), 0.5).exp_()
    if case["dtype"] == "float16":
        x *= 100.0  # float16 gradients are scaled
    return x.to(DTYPES[case["dtype"]])


def prepare(case: dict, seed: int) -> dict:
    if case["kind"] == "step":
        return _prepare_step(case, seed)
    if case["kind"] == "orthogonalize":
        return {"fn": newton_schulz_fn(NewtonSchulz(case["iteration"])), "x": _updates(case, seed)}
    g = torch.Generator(device="cuda").manual_seed(seed)
    stacks, shadows, sources = [], [], []
    for shape, count, _ in _shapes(case["shapes"]):
        shadow, source = _Stack(shape, count), _Stack(shape, count)
        source.whole.copy_(_normal(g, source.whole.shape, 0.02))
        shadow.whole.copy_(source.whole + _normal(g, source.whole.shape, 2e-3))
        stacks.append(shadow.whole)
        shadows += [shadow[i] for i in range(count)]
        sources += [source[i] for i in range(count)]
    return {"shadows": shadows, "sources": sources, "outputs": stacks}


def run(state: dict):
    if "opt" in state:
        state["opt"].step()
        return state["outputs"]
    if "fn" in state:
        return state["fn"](state["x"], NS_EPS)
    foreach_ema_update_(state["shadows"], state["sources"], decay=EMA_DECAY)
    return state["outputs"]


# ---- the same in float64 ---------------------------------------------------------------

def _coefficients(iteration: str) -> tuple[list[tuple[float, float, float]], float]:
    """The five steps' (a, b, c) and the factor on the input's norm."""
    if iteration == "gram":
        s = 1.05
        rows = [(8.28721201814563, -23.595886519098837, 17.300387312530933),
                (4.107059111542203, -2.9478499167379106, 0.5448431082926601),
                (3.9486908534822946, -2.908902115962949, 0.5518191394370137),
                (3.3184196573706015, -2.488488024314874, 0.51004894012372),
                (2.300652019954817, -1.6689039845747493, 0.4188073119525673)]
        return [(a / s, b / s ** 3, c / s ** 5) for a, b, c in rows], 1.0
    if iteration.startswith("polar"):
        return [(8.156554524902461, -22.48329292557795, 15.878769915207462),
                (4.042929935166739, -2.808917465908714, 0.5000178451051316),
                (3.8916678022926607, -2.772484153217685, 0.5060648178503393),
                (3.285753657755655, -2.3681294933425376, 0.46449024233003106),
                (2.3465413258596377, -1.7097828382687081, 0.42323551169305323)], 1.02
    return [(3.4445, -4.7750, 2.0315)] * 5, 1.0


def _polynomials(x: torch.Tensor, iteration: str) -> torch.Tensor:
    """The iteration's five polynomials of one matrix, through the Gram matrix of its short side."""
    rows, safety = _coefficients(iteration)
    tall = x.shape[0] > x.shape[1]
    x = x.double()
    x = (x.mT if tall else x).contiguous()
    x = x / (x.norm() * safety + NS_EPS)
    for a, b, c in rows:
        g = x @ x.mT
        p = c * (g @ g) + b * g
        x = a * x + p @ x
    return x.mT if tall else x


def _exact_block(case, w, g, m, v) -> None:
    """One block's step in float64, in place."""
    rows, cols = w.shape
    k = _selected(rows, case["fraction"])
    short = min(rows, cols)
    step = LR * 0.2 * math.sqrt(max(rows, cols)) * math.sqrt(short / min(k, cols))
    m += g
    if k < rows:
        at = m.abs().sum(1).topk(k).indices.sort().values
        u = m[at]
        m[at] = u * MOMENTUM
    else:
        at = torch.arange(rows, device=w.device)
        u = m.clone()
        m *= MOMENTUM
        if case["update"] == "muon":
            u = g + m
    o = _polynomials(u, case["iteration"])
    if case["update"] == "dion3":
        v[at] = v[at] * BETA2 + (1 - BETA2) * o.square().mean(1)
        n = o / (v[at].sqrt() + 1e-8)[:, None]
        o = n * (o.norm() / n.norm().clamp_min(1e-8))
    w *= 1 - LR * case["decay"]
    w[at] -= step * o


def _exact_step(case: dict, seed: int) -> dict:
    shapes, vectors = _lists(case)
    matrices, adamw = [], []
    for (shape, heads), count in shapes.items():
        m = {key: _Stack(shape, count) for key in ("wgs" if case["ema"] else "wg")}
        matrices.append({**m, "heads": heads or 1,
                         "m": torch.empty(count, *shape, device="cuda"),
                         "v": torch.empty(count, shape[0], device="cuda")})
    for shape, count, decayed in vectors:
        a = {key: _Stack(shape, count) for key in ("wgmvs" if case["ema"] else "wgmv")}
        adamw.append({**a, "decay": case["decay"] if decayed else 0.0})
    _fill(torch.Generator(device="cuda").manual_seed(seed), case, matrices, adamw)
    outputs = {}
    for i, s in enumerate((*matrices, *adamw)):
        for key in "wgmvs":
            if key in s:
                s[key] = (s[key].whole if isinstance(s[key], _Stack) else s[key]).double()
        if i < len(matrices):
            heads = s["heads"]
            rows, cols = s["w"].shape[1] // heads, s["w"].shape[2]
            per_block = [s[key].view(-1, rows, cols) for key in "wgm"] + [s["v"].view(-1, rows)]
            for w, g, m, v in zip(*per_block):
                _exact_block(case, w, g, m, v)
        else:
            t = ADAMW_STEPS + 1
            s["w"] *= 1 - LR * s["decay"]
            s["m"] += (1 - BETAS[0]) * (s["g"] - s["m"])
            s["v"] += (1 - BETAS[1]) * (s["g"].square() - s["v"])
            denominator = s["v"].sqrt() / math.sqrt(1 - BETAS[1] ** t) + EPS
            s["w"] -= LR / (1 - BETAS[0] ** t) * s["m"] / denominator
        if case["ema"]:
            s["s"] += (1 - EMA_DECAY) * (s["w"] - s["s"])
        s.pop("g")
        for key in "wmvs":
            if key in s:
                outputs["%d%s" % (i, key)] = s[key]
    return outputs


def exact(case: dict, seed: int):
    if case["kind"] == "step":
        return _exact_step(case, seed)
    if case["kind"] == "orthogonalize":
        return torch.stack([_polynomials(x, case["iteration"]) for x in _updates(case, seed)])
    state = prepare(case, seed)
    shadows = [s.double() for s in state["outputs"]]
    g = torch.Generator(device="cuda").manual_seed(seed)
    for shadow, (shape, count, _) in zip(shadows, _shapes(case["shapes"])):
        source = _normal(g, (count, *shape), 0.02)
        _normal(g, (count, *shape), 2e-3)
        shadow += (1 - EMA_DECAY) * (source.double() - shadow)
    return shadows
