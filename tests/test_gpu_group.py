"""The first stage of rows over 32 elements (csrc/ti_group.hip: a workgroup builds the hull of a
group of up to 16384 elements) on the GPU against the oracle, at the sizes where its shapes
change (threads a group, elements a thread, groups a row) and on the data that decides its paths:
few candidates, more candidates than its slots (chunks merged by reference), exact ties, a point
far below that takes a whole convex chain with it, values that put the rounding margin over
every height, NaN rows. Fits, start bits and both gradients."""

from __future__ import annotations

import numpy as np
import pytest

import oracle
from gpu_util import check_fit, gpu_fit, tolerance
from test_gpu_tiles import gpu_grads
from torchisotonic_amd import _ext

pytestmark = pytest.mark.gpu

# a wave of 4, 8 elements a thread; two waves; 256 threads of 8, 16; 512 of 16, 32 (float64 1024 of
# 16); one past each, where a thread, a wave or a shape more begins; two groups and more a row
SIZES = [33, 255, 257, 511, 513, 1023, 1025, 2047, 2049, 4095, 4097, 5000, 8191, 8193, 16383, 16385, 33000]


def rows(kind: str, n: int, rng: np.random.Generator) -> np.ndarray:
    i = np.arange(n)
    if kind == "noise":
        return np.linspace(0, 3, n) + rng.standard_normal(n)
    if kind == "rise":  # a vertex at every element
        return 1e-3 * i + rng.random()
    if kind == "cliff":  # a convex chain, all of it pooled by its last element
        return np.r_[1e-3 * i[:-1], -1e3 * n]
    if kind == "drops":  # near-monotone, several chains pooled back
        return 1e-3 * i + 1e-5 * rng.standard_normal(n) - 0.3 * (i % 997 == 996)
    if kind == "ties":  # every sum an exact integer
        return rng.integers(0, 3, n).astype(float)
    assert kind == "mixed"  # magnitudes that put the margin over every other height
    return np.where(i == n // 3, 1e25, rng.standard_normal(n))


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_groups(n: int, weighted: bool, dtype: type) -> None:
    print(f"groups n={n} weighted={weighted} {np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(n + weighted)
    kinds = ["noise", "rise", "cliff", "drops", "ties"]
    y = np.stack([rows(k, n, rng) for k in kinds] + [rows("noise", n, rng)])
    y[-1, n // 2] = np.nan
    y = y.astype(dtype)
    w = None
    if weighted:
        w = rng.random(y.shape) + 0.1
        w[4] = rng.integers(1, 5, n)
        w = w.astype(dtype)
    # (float32's running sums round differently on the cliff than the oracle's float64 ones)
    check_fit(y, w, check_starts=True)
    check_fit(y, w, increasing=False, y_min=-0.5, y_max=2.0)
    g = rng.standard_normal(y.shape).astype(dtype)
    gs, _ = gpu_grads(y, w, g)
    ok = slice(0, 5)
    w64 = None if w is None else w[ok].astype(np.float64)
    fit, st = oracle.pava(y[ok], None if w is None else w[ok], acc="f64")
    ey, ew = oracle.block_grad(st, g[ok].astype(np.float64), w64, y[ok].astype(np.float64), fit, want_w=weighted)
    tol = 1e-12 if dtype == np.float64 else 2e-5
    np.testing.assert_allclose(gs[0][ok], ey, rtol=tol, atol=tol)
    if weighted:
        scale = 1 + np.abs(y[ok] - fit).max(axis=1, keepdims=True)
        np.testing.assert_allclose(gs[1][ok] / scale, ew / scale, rtol=tol, atol=tol)


@pytest.mark.parametrize("n", [200, 3000, 20_000])
def test_margin_over_every_height(n: int) -> None:
    # one value so large that the margin drops nothing by chords: every rise is a candidate, and
    # the exact neighbour tests decide. Before the value, whose sums it is not in, fit and start
    # bits are exact to those elements' own magnitude; from it on sums round the others away.
    rng = np.random.default_rng(n)
    for dtype in (np.float32, np.float64):
        y = np.stack([rows("mixed", n, rng) for _ in range(3)]).astype(dtype)
        got, starts = gpu_fit(y)
        want, want_starts = oracle.pava(y.astype(np.float64), acc="f64")
        assert float(np.abs(got - want).max()) <= 4 * np.finfo(dtype).eps * 1e25
        before = slice(0, n // 3)
        assert float(np.abs(got - want)[:, before].max()) <= tolerance(y[:, before])
        np.testing.assert_array_equal(starts[:, : n // 3 + 1], want_starts[:, : n // 3 + 1])


@pytest.mark.parametrize(("n", "batches"), [(1100, (4, 3000)), (2001, (4, 3000)), (2500, (4, 132, 600)),
                                            (9001, (4, 40, 72, 132, 600)), (16384, (4, 20, 260)), (33_000, (4, 100))])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_overflowing_groups_shared_by_workgroups(n: int, batches: tuple[int, ...], dtype: type) -> None:
    # A group of more candidates than slots is built by one workgroup or, where groups are few, by
    # several that share its chunks: as many as chunks for 4 rows, two or three of them for up to 128
    # groups, one from 256 on. The same rows give the same bits whoever builds them, and the oracle's.
    print(f"overflowing groups n={n} {np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(n)
    y = np.stack([rows(k, n, rng) for k in ("rise", "drops", "noise", "rise")]).astype(dtype)
    w = (rng.random(y.shape) + 0.1).astype(dtype)
    for ww in (None, w):
        first = None
        for b in batches:
            if _ext.geometry(b, n, ww is not None) != _ext.geometry(4, n, ww is not None):
                first = None  # (other groups: compared with the oracle only)
            got, starts = check_fit(np.tile(y, (b // 4, 1)), None if ww is None else np.tile(ww, (b // 4, 1)))
            assert (np.diff(got, axis=1) >= 0).all()
            if first is None:
                first = got[:4], starts[:4]
            np.testing.assert_array_equal(got, np.tile(first[0], (b // 4, 1)))
            np.testing.assert_array_equal(starts, np.tile(first[1], (b // 4, 1)))


def test_overflowing_groups_replayed() -> None:
    # the count of a group's workgroups starts from zero in every replay of a captured call, whether
    # the group overflowed in the replay before or not
    import torch

    import torchisotonic_amd

    print("overflowing groups in a graph", flush=True)
    n = 9001
    rng = np.random.default_rng(4)
    data = [np.stack([rows(k, n, rng) for k in kinds]) for kinds in
            (("rise", "drops", "rise"), ("noise", "rise", "noise"), ("rise", "rise", "drops"), ("noise", "noise", "noise"))]
    data = [torch.from_numpy(d.astype(np.float32)).cuda() for d in data]
    y = data[0].clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torchisotonic_amd.isotonic(y)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fit = torchisotonic_amd.isotonic(y)
    for k in (0, 0, 1, 3, 2, 0):
        y.copy_(data[k])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(fit, torchisotonic_amd.isotonic(data[k]))


@pytest.mark.parametrize("n", [200, 512, 2048, 3840, 5000, 16384, 33_000])
@pytest.mark.parametrize("weighted", [False, True])
def test_sums_over_threads_carry_their_rounding(n: int, weighted: bool) -> None:
    # Pairs 2^60, -2^60 on either side of a multiple of 32 (so never in one thread's elements, whose
    # sum is a float64), the rest of their two threads' elements 0: each pair cancels exactly, and
    # beside it the sums across threads keep the other elements' parts, nine orders under 2^60's
    # last place, only with their rounding errors. Increasing rows pool a pair and its zeros; the
    # fit elsewhere is that of the row with the pair put to 0.
    rng = np.random.default_rng(n)
    y = (np.linspace(-1, 1, n) + rng.standard_normal((4, n))).astype(np.float32)
    for row in y:
        for m in [m for m in rng.permutation(np.arange(1, n // 32)) if m % 64 != 0][: max(1, n // 256)]:
            row[32 * m - 32:32 * m + 32] = 0
    plain = y.copy()
    for r, row in enumerate(y):
        # (every second run of 64 zeros; none across groups, whose points are float64s from its start)
        at = [m for m in range(1, n // 32) if m % 64 != 0 and not row[32 * m - 32:32 * m + 32].any()]
        for m in at[::2]:
            row[32 * m - 1], row[32 * m] = 2.0**60, -(2.0**60)
    w = (rng.random(y.shape) + 0.1).astype(np.float32) if weighted else None
    if weighted:
        w[y != plain] = 1
    got, _ = gpu_fit(y, w)
    want, _ = oracle.pava(plain, w, acc="f64")
    assert (y != plain).any()
    assert float(np.abs(got - want).max()) <= 4 * 2.0**-23 * float(np.abs(plain).max())


def test_ragged_rows_end_where_they_end() -> None:
    # rows read in place up to their own length, the block's rest one block of pad: lengths around
    # the shapes' edges in one bucket, and rising rows that overflow it
    import torch

    import torchisotonic_amd

    rng = np.random.default_rng(3)
    lens = np.r_[[4100, 5000, 6143, 6144, 6145, 8191, 8192] * 3, np.full(20, 7000)]
    off = np.r_[0, np.cumsum(lens)]
    y = np.concatenate([rows("rise" if k % 3 == 0 else "noise", m, rng) for k, m in enumerate(lens)]).astype(np.float32)
    for inc in (True, False):
        fit = torchisotonic_amd.isotonic_ragged(torch.from_numpy(y).cuda(), torch.from_numpy(off).cuda(), increasing=inc)
        got = fit.cpu().numpy()
        for k in range(len(lens)):
            row = y[off[k]:off[k + 1]][None]
            want, _ = oracle.pava(row, increasing=inc, acc="f64")
            assert float(np.abs(got[off[k]:off[k + 1]] - want[0]).max()) <= 4 * 2.0**-23 * np.abs(row).max()


def test_one_group_a_row() -> None:
    # rows of up to 16384 elements are one group however few they are; longer rows are not
    for n in (2049, 16384):
        assert _ext.geometry(1, n, False)["levels"] == 1
    assert _ext.geometry(1, 16385, False)["levels"] == 2
