"""Dense similarities as they come in earnest: masks of the worst value or of
the type's lowest number, negated distances (-0 where they are zero), and sums
that leave float32: scores and paths against the oracle."""

import numpy as np
import pytest

import oracle as O
import pyalign_amd as pa
from tests.test_gpu_band import LOCS, lengths, make_solver

pytestmark = pytest.mark.gpu

HUGE = float(np.finfo(np.float32).max)


def similarities(rng, kind, a, b):
    S = rng.integers(-2, 4, (a, b)).astype(np.float32)
    if kind in ("worst", "lowest"):
        S[rng.random((a, b)) < 0.3] = -np.inf if kind == "worst" else -HUGE
    elif kind == "distances":
        S = -np.abs(rng.integers(0, 4, (a, 1)) - rng.integers(0, 4, (1, b))).astype(np.float32)
    elif kind == "zeros":  # (-0 along the diagonal from the corner, where cells tie with gaps)
        S[rng.random((a, b)) < 0.4] = -0.0
        np.fill_diagonal(S, -0.0)
    else:
        S[rng.random((a, b)) < 0.2] = HUGE
    return S


@pytest.mark.parametrize("loc", list(LOCS))
@pytest.mark.parametrize("direction", ["maximize", "minimize"])
@pytest.mark.parametrize("kind", ["worst", "lowest", "distances", "zeros", "overflow"])
@pytest.mark.parametrize("short", [False, True])  # (columns: rows staged in LDS, or not)
def test_dense(loc, direction, kind, short):
    rng = np.random.default_rng(len(loc) + len(kind))
    n = 50
    ls, lt = lengths(rng, n, 1, 80, 3 if short else 8, 80)
    ls[:2], lt[:2] = (600, 64), (40, 300)
    S = [similarities(rng, kind, a, b) * (1 if direction == "maximize" else -1) for a, b in zip(ls, lt)]
    off = np.concatenate([[0], np.cumsum(ls.astype(np.int64) * lt)[:-1]])
    odir = O.MAXIMIZE if direction == "maximize" else O.MINIMIZE
    for gap in (("affine", 5, 1), ("affine", 3, 0), ("linear", 2)):
        got = make_solver(loc, gap, direction, pa.Solution, 1024, 512).solve_ragged(
            "solution", "dense", ls, lt, dense=np.concatenate([x.ravel() for x in S]), dense_off=off)
        for k in range(n):
            with np.errstate(all="ignore"):
                ref = O.OracleResult(O.make_config(locality=LOCS[loc][1], direction=odir, gap=gap, goal=O.GOAL_ONE,
                                                   lim_s=1024, lim_t=512), S[k])
            if not ref.has_seed:
                assert got[k].score is None, k
                continue
            assert np.float32(got[k].score).tobytes() == ref.score.tobytes(), (k, gap)
            assert np.array_equal(np.asarray(got[k].path, np.int32), ref.path()), (k, gap)
