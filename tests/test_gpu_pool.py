"""Equal sorted keys pooled into one point each (csrc/ti_calib.hip, ti_pool) against numpy in long
double: runs of one element, of a few, of several tiles and of the whole input, sizes at the edges
of a step (64 elements) and a tile (1024), each dtype, a NaN kept to its own run.

Tolerance: an element's value is added at most 6 times within its step, 16 times from step to step
of its tile, and 6 + 4 times over the tiles of its run (195 tiles, 64 a round), each sum rounded
once, as are its product with the weight and the division; the weights' sum likewise. So the mean
is within 2 * 34 * 2^-53 of sum(|w y|) / sum(w).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from torchisotonic_amd import _ext

pytestmark = pytest.mark.gpu


def say(what: str) -> None:
    print(what, flush=True)


def runs_of(kind: str, n: int, rng: np.random.Generator) -> np.ndarray:
    if kind == "single":
        return np.arange(n)
    if kind == "equal":
        return np.zeros(n, dtype=np.int64)
    mean = {"pairs": 1.3, "short": 9.0, "long": 3000.0}[kind]
    return np.cumsum(rng.random(n) < 1.0 / mean)


@pytest.mark.parametrize("keys_dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["single", "pairs", "short", "long", "equal"])
def test_runs_against_long_double(kind: str, dtype, keys_dtype) -> None:
    for n in (1, 2, 63, 64, 65, 1023, 1024, 1025, 4096, 70_001, 200_000):
        rng = np.random.default_rng(n)
        run = runs_of(kind, n, rng)
        run -= run[0]
        keys = run.astype(keys_dtype) - 7
        order = rng.permutation(n)
        y = rng.normal(size=n).astype(dtype)
        for w in (None, rng.uniform(0.1, 2.0, n).astype(dtype)):
            say(f"pool {kind} n={n} {np.dtype(dtype)} keys {np.dtype(keys_dtype)} weighted={w is not None}")
            xp, mean, weight, inverse = _ext.pool_sorted(
                torch.from_numpy(keys).cuda(), torch.from_numpy(order).cuda(), torch.from_numpy(y).cuda(),
                None if w is None else torch.from_numpy(w).cuda(), True)
            ys = y[order].astype(np.longdouble)
            ws = np.ones(n, np.longdouble) if w is None else w[order].astype(np.longdouble)
            first = np.flatnonzero(np.r_[True, run[1:] != run[:-1]])
            total = np.add.reduceat(ws, first)
            want = np.add.reduceat(ws * ys, first) / total
            bound = 68 * 2.0**-53
            np.testing.assert_array_equal(xp.cpu().numpy(), keys[first].astype(np.float64))
            np.testing.assert_array_equal(inverse.cpu().numpy(), run)
            assert (np.abs(weight.cpu().numpy() - total) <= bound * total).all()
            assert (np.abs(mean.cpu().numpy() - want) <= bound * np.add.reduceat(ws * np.abs(ys), first) / total).all()


def test_a_nan_value_stays_in_its_run_and_nan_keys_apart() -> None:
    say("pool NaN")
    n = 5000
    keys = torch.arange(n, dtype=torch.float64, device="cuda").div(50, rounding_mode="floor")
    keys[-3:] = float("nan")
    y = torch.ones(n, device="cuda")
    y[1075] = float("nan")
    y[4000] = float("inf")
    xp, mean, weight, inverse = _ext.pool_sorted(keys, torch.arange(n, device="cuda"), y, None, False)
    assert inverse is None and xp.numel() == 103 and bool(xp[-3:].isnan().all())
    want = torch.ones(103, dtype=torch.float64, device="cuda")
    want[21], want[80] = float("nan"), float("inf")
    torch.testing.assert_close(mean, want, rtol=0, atol=0, equal_nan=True)
    assert weight[:99].eq(50).all() and weight[99] == 47 and weight[-3:].eq(1).all()


@pytest.mark.parametrize("bad", [0.0, -1.0, float("nan")])
@pytest.mark.parametrize("at", [0, 1024, 2999])
def test_a_weight_that_is_not_positive_is_refused(bad: float, at: int) -> None:
    say(f"pool weight {bad} at {at}")
    w = torch.ones(3000, device="cuda")
    w[at] = bad
    keys, order = torch.arange(3000.0, device="cuda"), torch.arange(3000, device="cuda")
    with pytest.raises(ValueError, match="strictly positive"):
        _ext.pool_sorted(keys, order, torch.ones_like(w), w, False)


def test_gradients_flow_through_the_calibration_fit() -> None:
    say("calibration gradient")
    from torchisotonic_amd.calibration import calibration_fit

    keys = torch.tensor([1.0, 1.0, 2.0, 3.0], device="cuda")
    y = torch.tensor([3.0, 1.0, 1.0, 5.0], device="cuda", requires_grad=True)
    xp, fp = calibration_fit(keys, y)
    fp.sum().backward()
    # blocks {1, 2} (weights 2 and 1, two knots) and {3}: d(sum fp)/dy = 2/3 each, then 1
    torch.testing.assert_close(y.grad, torch.tensor([2 / 3, 2 / 3, 2 / 3, 1.0], device="cuda"))
    with torch.no_grad():
        torch.testing.assert_close(calibration_fit(keys, y)[1], fp.detach(), rtol=0, atol=1e-15)
