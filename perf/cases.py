"""The workloads this package is timed on, as a user's program calls them: fits and their
gradients over rows from one small calibration set to a single row of 1e8 elements, ragged rows,
soft ranks, and calibration fit and predict.

``listed()`` gives the fixed workloads and ``draw(rng)`` more of the same ranges; ``prepare``
makes a workload's inputs on the GPU from a seed, ``run`` makes one pass through the package's
public functions and returns every output, ``work`` counts the bytes and operations no
implementation can do without, and ``exact`` restates the results in float64 with torch's own
operators (pool adjacent violators over whole runs at a time).
"""

from __future__ import annotations

import math
import random

import torch

import torchisotonic_amd

DTYPES = {"float32": torch.float32, "float64": torch.float64}

# ``kind``: "rows" (dense rows of one length), "ragged", "soft_rank", "calibrate".
# ``data`` of dense and ragged rows:
#   "trend"      step * i + N(0, 1), the sign of step that of the fit's direction
#   "sigmoid"    sigmoid(linspace(-4, 4) + N(0, 0.5)), probabilities still noisy
#   "labels"     0/1 labels of sorted scores, P(1) = sigmoid(score)
# ``weight``: "" (none), "uniform" (U(0, 1) + 0.1), "counts" (integers 1..5), "exponential"
# (Bayesian bootstrap weights, floored at 1e-6). ``grad``: "" (forward only), "y", "yw".


def _rows(name: str, batch: int, n: int, **kw) -> dict:
    case = {"kind": "rows", "batch": batch, "n": n, "dtype": "float32", "data": "trend", "weight": "",
            "increasing": True, "clamp": False, "grad": "", **kw}
    return {"name": name, **case} if name else case


def listed() -> list[dict]:
    return [
        # One small calibration set (a validation split's scores and labels, sorted): the call
        # whose time is the host's path and the launches.
        _rows("one_row_500", 1, 500, data="labels", weight="uniform", clamp=True),
        # Many short dose-response or quantile rows, the package's headline workload.
        _rows("rows_16", 1_000_000, 16, increasing=False),
        # A layer over short rows in training, weighted, of an odd length.
        _rows("rows_27_train", 200_003, 27, weight="uniform", grad="yw"),
        # A monotone layer over a few hundred ordered bins, in training.
        _rows("rows_200_train", 20_000, 200, grad="y"),
        # A batch of curves of a thousand points.
        _rows("rows_1000", 10_000, 1000, increasing=False),
        # A thousand noisy series of 5000 points.
        _rows("rows_5000", 1000, 5000),
        # The same size in float64: weighted probabilities clamped to [0, 1], with both gradients.
        _rows("rows_5000_f64_train", 1000, 5000, dtype="float64", data="sigmoid", weight="uniform",
              increasing=False, clamp=True, grad="yw"),
        # Bayesian bootstrap of one calibration curve: shared labels, weights of each row's own.
        _rows("bootstrap_65536_train", 1000, 65536, data="labels", weight="exponential", grad="yw"),
        # Calibration of 1e8 scored impressions in one row, repeated scores already counted.
        _rows("one_row_1e8", 1, 100_000_000, data="labels", weight="counts"),
        # Per-group fits of groups of very different sizes, in training.
        {"name": "ragged_2000_train", "kind": "ragged", "rows": 100_000, "shortest": 1, "longest": 2000,
         "weight": "", "increasing": True, "grad": "y"},
        # Soft ranks as a loss over lists of 10000.
        {"name": "soft_rank_10000_train", "kind": "soft_rank", "batch": 64, "n": 10_000, "strength": 1.0},
        # Calibrating a click model on a day of scores, then mapping as many new ones.
        {"name": "calibrate_6500000", "kind": "calibrate", "scores": 6_500_000},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choices(("rows", "ragged", "soft_rank", "calibrate"), (12, 2, 1, 1))[0]
    if kind == "ragged":
        longest = _log_int(rng, 8, 4000)
        return {"kind": kind, "rows": _log_int(rng, 500, max(501, min(300_000, 20_000_000 // longest))),
                "shortest": rng.randint(1, longest), "longest": longest, "weight": rng.choice(("", "uniform")),
                "increasing": rng.random() < 0.5, "grad": rng.choice(("", "y"))}
    if kind == "soft_rank":
        n = _log_int(rng, 20, 200_000)
        return {"kind": kind, "batch": _log_int(rng, 1, max(2, 1_000_000 // n)), "n": n,
                "strength": rng.choice((1.0, 0.1, 1.0 / n))}
    if kind == "calibrate":
        return {"kind": kind, "scores": _log_int(rng, 1000, 6_500_000)}
    n = _log_int(rng, 2, 20_000_000)
    batch = _log_int(rng, 1, max(2, min(1_000_000, 20_000_000 // n)))
    data = rng.choice(("trend", "trend", "sigmoid", "labels"))
    return _rows("", batch, n, dtype=rng.choice(("float32", "float32", "float32", "float64")), data=data,
                 weight=rng.choice(("", "uniform", "counts", "exponential")), increasing=rng.random() < 0.6,
                 clamp=data != "trend" and rng.random() < 0.5, grad=rng.choice(("", "y", "yw")))


# --- inputs -----------------------------------------------------------------------------------


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _weights(kind: str, shape: tuple[int, ...], dtype: torch.dtype, gen: torch.Generator) -> torch.Tensor | None:
    if kind == "":
        return None
    if kind == "counts":
        return torch.randint(1, 6, shape, generator=gen, device="cuda").to(dtype)
    if kind == "uniform":
        return torch.rand(shape, generator=gen, device="cuda", dtype=dtype) + 0.1
    return torch.empty(shape, device="cuda", dtype=dtype).exponential_(generator=gen).clamp_(min=1e-6)


def _values(case: dict, gen: torch.Generator) -> torch.Tensor:
    batch, n, dtype = case["batch"], case["n"], DTYPES[case["dtype"]]
    sign = 1.0 if case["increasing"] else -1.0
    if case["data"] == "trend":
        # 0.1 a step in short rows, 5 in all in long ones, as curves have
        step = sign * min(0.1, 5.0 / n)
        y = torch.randn(batch, n, generator=gen, device="cuda", dtype=dtype)
        return y.add_(torch.arange(n, device="cuda", dtype=dtype), alpha=step)
    if case["data"] == "sigmoid":
        y = torch.randn(batch, n, generator=gen, device="cuda", dtype=dtype).mul_(0.5)
        return y.add_(sign * torch.linspace(-4, 4, n, device="cuda", dtype=dtype)).sigmoid_()
    if batch == 1:
        score = (torch.randn(n, generator=gen, device="cuda") * 1.5).sort().values * sign
        return (torch.rand(n, generator=gen, device="cuda") < score.sigmoid()).to(dtype).view(1, n)
    score = torch.linspace(-4, 4, n, device="cuda") * sign
    y = (torch.rand(n, generator=gen, device="cuda") < score.sigmoid()).to(dtype)
    return y.expand(batch, n).contiguous()


def _clicks(m: int, gen: torch.Generator) -> tuple[torch.Tensor, torch.Tensor]:
    """m float32 click probabilities, one in 13 a repeat of another (as a day's scores repeat),
    and labels of a model that is off by a slope and a shift. The distinct scores are pushed
    apart by single float32 steps, so that every seed has the same number of knots."""
    k = m - m // 13
    logit = (torch.randn(k, generator=gen, device="cuda", dtype=torch.float64) * 1.5 - 1.2).sort().values
    at = torch.arange(k, device="cuda")
    bits = torch.cummax(logit.sigmoid().float().view(torch.int32).long() - at, 0).values + at
    score = bits.int().view(torch.float32)
    again = torch.randint(0, k, (m - k,), generator=gen, device="cuda")
    score = torch.cat([score, score[again]])[torch.randperm(m, generator=gen, device="cuda")]
    draws = torch.rand(m, generator=gen, device="cuda", dtype=torch.float64)
    return score, (draws < (score.double().logit() * 0.8 + 0.3).sigmoid()).float()


def _lengths(case: dict) -> torch.Tensor:
    lo, span = case["shortest"], case["longest"] + 1 - case["shortest"]
    return lo + torch.arange(case["rows"], device="cuda") * span // case["rows"]


def prepare(case: dict, seed: int) -> dict:
    gen = _generator(seed)
    if case["kind"] == "calibrate":
        scores, labels = _clicks(case["scores"], gen)
        return {"case": case, "scores": scores, "labels": labels, "queries": _clicks(case["scores"], gen)[0]}
    if case["kind"] == "soft_rank":
        shape = (case["batch"], case["n"])
        x = torch.randn(shape, generator=gen, device="cuda")
        return {"case": case, "y": x.requires_grad_(), "g": torch.randn(shape, generator=gen, device="cuda")}
    if case["kind"] == "ragged":
        # lengths spread evenly from the shortest to the longest, in an order of the seed's own
        lengths = _lengths(case)[torch.randperm(case["rows"], generator=gen, device="cuda")]
        offsets = torch.zeros(case["rows"] + 1, dtype=torch.int64, device="cuda")
        torch.cumsum(lengths, 0, out=offsets[1:])
        total = int(offsets[-1])
        y = torch.randn(total, generator=gen, device="cuda")
        first = torch.repeat_interleave(offsets[:-1], lengths, output_size=total)
        y.add_(torch.arange(total, device="cuda") - first, alpha=0.001 if case["increasing"] else -0.001)
        state = {"case": case, "offsets": offsets, "y": y, "w": _weights(case["weight"], (total,), y.dtype, gen)}
    else:
        y = _values(case, gen)
        state = {"case": case, "y": y, "w": _weights(case["weight"], tuple(y.shape), y.dtype, gen)}
    if case["grad"]:
        state["g"] = torch.randn(y.shape, generator=gen, device="cuda", dtype=y.dtype)
        y.requires_grad_()
        if case["grad"] == "yw" and state["w"] is not None:
            state["w"].requires_grad_()
    return state


# --- one pass ---------------------------------------------------------------------------------


def run(state: dict):
    case = state["case"]
    if case["kind"] == "calibrate":
        cal = torchisotonic_amd.IsotonicCalibrator().fit(state["scores"], state["labels"])
        return {"knots": cal.xp, "values": cal.fp, "predicted": cal.predict(state["queries"])}
    y, w = state["y"], state.get("w")
    if case["kind"] == "soft_rank":
        fit = torchisotonic_amd.soft_rank(y, case["strength"])
    elif case["kind"] == "ragged":
        fit = torchisotonic_amd.isotonic_ragged(y, state["offsets"], weight=w, increasing=case["increasing"])
    else:
        lo, hi = (0.0, 1.0) if case["clamp"] else (None, None)
        fit = torchisotonic_amd.isotonic(y, w, increasing=case["increasing"], y_min=lo, y_max=hi)
    inputs = [t for t in (y, w) if t is not None and t.requires_grad]
    if not inputs:
        return [fit]
    return [fit.detach(), *torch.autograd.grad(fit, inputs, state["g"])]


def _elements(case: dict) -> int:
    if case["kind"] == "ragged":
        return case["rows"] * (case["shortest"] + case["longest"]) // 2  # (to within one a row)
    return case["batch"] * case["n"]


def work(case: dict) -> dict:
    """Bytes: every input read once, every output written once. Operations: four an element for
    the sums and one hull test of a forward, three for the block sums and products of a backward;
    soft ranks and calibration sort too (a comparison an element and level)."""
    if case["kind"] == "calibrate":
        m = case["scores"]
        # scores, labels and queries in (4 B each), knots and values out (8 B each, nearly one a
        # score), predictions out (8 B)
        return {"bytes": 36 * m, "flops": m * (4 + 2 * math.log2(m))}
    e = _elements(case)
    if case["kind"] == "soft_rank":
        return {"bytes": 16 * e, "flops": e * (7 + math.log2(case["n"]))}
    size = 8 if case.get("dtype") == "float64" else 4
    tensors = 2 + bool(case["weight"])  # y (w) in, the fit out
    flops = 4
    if case["grad"]:
        tensors += 2  # g in, y's gradient out
        flops += 3
        if case["grad"] == "yw" and case["weight"]:
            tensors += 1
            flops += 2
    offsets = 8 * (case["rows"] + 1) if case["kind"] == "ragged" else 0
    return {"bytes": tensors * size * e + offsets, "flops": flops * e}


def tolerance(case: dict) -> dict:
    """About four times the largest difference from ``exact`` seen over the ranges drawn here
    (float32 results are float64 sums rounded once: 2e-8 to 2e-7; float64: up to 2e-15, more
    where sums cancel), per element about ten times that."""
    if case["kind"] == "calibrate":
        return {"rel": 1e-14, "max": 1e-12}  # float64 throughout; the knots are the scores themselves
    if case.get("dtype") == "float64":
        return {"rel": 1e-13, "max": 1e-11}
    return {"rel": 1e-6, "max": 1e-5}


# --- the same results in float64 --------------------------------------------------------------


def _pool(y: torch.Tensor, w: torch.Tensor, row: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Pool adjacent violators of the increasing fit of rows laid end to end: each pass pools
    every maximal run of blocks whose means do not rise, until none is left. Returns each
    element's block, and the blocks' means and weights."""
    sums, weights, block = y * w, w, None
    while True:
        means = sums / weights
        starts = torch.ones_like(row, dtype=torch.bool)
        starts[1:] = (means[1:] > means[:-1]) | (row[1:] != row[:-1])
        if bool(starts.all()):
            if block is None:
                block = torch.arange(y.numel(), device=y.device)
            return block, means, weights
        into = torch.cumsum(starts, 0) - 1
        count = int(into[-1]) + 1
        sums = torch.zeros(count, dtype=sums.dtype, device=y.device).index_add_(0, into, sums)
        weights = torch.zeros(count, dtype=sums.dtype, device=y.device).index_add_(0, into, weights)
        row = row[starts]
        block = into if block is None else into[block]


def _fit64(y, w, row, g, increasing, clamp, want_w):
    """The fit and gradients of flat rows: [fit, gy, gw], a gradient None where not wanted."""
    sign = 1.0 if increasing else -1.0
    y = y.detach().double()
    w = torch.ones_like(y) if w is None else w.detach().double()
    block, means, weights = _pool(sign * y, w, row)
    raw = (sign * means)[block]
    fit = raw.clamp(0.0, 1.0) if clamp else raw
    if g is None:
        return [fit]
    g = g.double() * ((raw >= 0.0) & (raw <= 1.0)) if clamp else g.double()
    share = (torch.zeros_like(means).index_add_(0, block, g) / weights)[block]
    return [fit, w * share, *([(y - raw) * share] if want_w else [])]


def exact(case: dict, seed: int):
    s = prepare(case, seed)
    if case["kind"] == "calibrate":
        return _calibrate64(s["scores"], s["labels"], s["queries"])
    if case["kind"] == "soft_rank":
        return _soft_rank64(s["y"].detach().double(), s["g"].double(), case["strength"])
    y, w, g = s["y"], s["w"], s.get("g")
    if case["kind"] == "ragged":
        lengths = s["offsets"].diff()
        row = torch.repeat_interleave(torch.arange(case["rows"], device="cuda"), lengths)
        clamp, shape = False, y.shape
    else:
        row = torch.arange(case["batch"], device="cuda").repeat_interleave(case["n"])
        clamp, shape = case["clamp"], y.shape
    flat = [None if t is None else t.reshape(-1) for t in (y, w, g)]
    out = _fit64(flat[0], flat[1], row, flat[2], case["increasing"], clamp, w is not None and w.requires_grad)
    return [t.view(shape) for t in out]


def _soft_rank64(x, g, strength):
    batch, n = x.shape
    s, perm = torch.sort(x / strength, dim=-1, descending=True)
    z = s - torch.arange(n, 0, -1, dtype=x.dtype, device=x.device)
    row = torch.arange(batch, device="cuda").repeat_interleave(n)
    dual, avg = _fit64(z.reshape(-1), None, row, g.gather(-1, perm).reshape(-1), False, False, False)
    rank = torch.empty_like(x).scatter_(-1, perm, s - dual.view(batch, n))
    back = torch.empty_like(x).scatter_(-1, perm, avg.view(batch, n))
    # below a strength of 1 float32's rounding of x / strength decides which neighbours pool, and
    # the gradient jumps where they do
    return [rank, (g - back) / strength if strength >= 1.0 else None]


def _calibrate64(scores, labels, queries):
    knots, into, counts = torch.unique(scores.double(), return_inverse=True, return_counts=True)
    counts = counts.double()
    sums = torch.zeros_like(knots).index_add_(0, into, labels.double())
    block, means, _ = _pool(sums / counts, counts, torch.zeros_like(knots, dtype=torch.int64))
    values = means[block]
    q = queries.double()
    at = torch.searchsorted(knots, q).clamp(1, max(1, knots.numel() - 1))
    lo, hi = at - 1, at.clamp(max=knots.numel() - 1)
    t = ((q - knots[lo]) / (knots[hi] - knots[lo]).clamp(min=1e-300)).clamp(0.0, 1.0)
    return {"knots": knots, "values": values, "predicted": values[lo] + t * (values[hi] - values[lo])}
