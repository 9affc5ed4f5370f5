"""Gap costs and similarities that max / min folds cannot take (infinite costs,
sums beyond float32) and those at the edge of what they can (similarities of
the type's lowest value): scores and paths against the oracle, by every form
that folds."""

import zlib

import numpy as np
import pytest

import oracle as O
import pyalign_amd as pa
from tests.test_gpu_band import LOCS, dense_of, lengths, make_solver, ragged_codes

pytestmark = pytest.mark.gpu

HUGE = float(np.finfo(np.float32).max)
INF = float("inf")
# name: (gap, similarities of a match and of mismatches, maximising)
VALUES = {"infinite open": (("affine", INF, 1), (2.0, -1.0)),
          "infinite linear": (("linear", INF), (2.0, -1.0)),
          "sums overflow": (("affine", 3, 1), (HUGE, -HUGE)),
          "lowest": (("affine", 3, 1), (2.0, -HUGE)),
          "huge costs": (("affine", 1e30, 1e30), (1e30, -1e30))}


# (global, infinite linear: 0 * inf makes the corner of the borders NaN)
@pytest.mark.parametrize("loc,values", [(x, v) for x in LOCS for v in VALUES if (x, v) != ("global", "infinite linear")])
@pytest.mark.parametrize("direction", ["maximize", "minimize"])
@pytest.mark.parametrize("form", ["indexed", "binary"])
def test_values(loc, values, direction, form):
    gap, (eq, ne) = VALUES[values]
    if direction == "minimize":
        eq, ne = -eq, -ne
    rng = np.random.default_rng(zlib.crc32(repr((loc, values, direction, form)).encode()))
    ls, lt = lengths(rng, 40, 1, 30, 1, 30)
    ls[0], lt[0] = 600, 70
    cs, ct, os_, ot = ragged_codes(rng, ls, lt, 4)
    payload = dict(off_s=os_, off_t=ot)
    table = np.full((4, 4), ne, np.float32)
    np.fill_diagonal(table, eq)
    if form == "binary":
        payload.update(codes_s=cs.astype(np.uint32), codes_t=ct.astype(np.uint32), eq=eq, ne=ne)
    else:
        payload.update(codes_s=cs, codes_t=ct, table=table)
    odir = O.MAXIMIZE if direction == "maximize" else O.MINIMIZE
    for codomain, kind, goal in ((pa.Score, "score", O.GOAL_SCORE), (pa.Solution, "solution", O.GOAL_ONE)):
        got = make_solver(loc, gap, direction, codomain, 1024, 128).solve_ragged(kind, form, ls, lt, **payload)
        for k in range(len(ls)):
            S = dense_of(form, k, cs, ct, os_, ot, ls, lt, table, eq, ne)
            ref = O.OracleResult(O.make_config(locality=LOCS[loc][1], direction=odir, gap=gap, goal=goal, lim_s=1024,
                                               lim_t=128), S)
            if kind == "solution" and not ref.has_seed:
                assert got[k].score is None
                continue
            score = got[k] if kind == "score" else got[k].score
            assert np.array_equal(np.float32(score), ref.score, equal_nan=True), (k, score, ref.score)
            if kind == "solution":
                assert np.array_equal(np.asarray(got[k].path, np.int32), ref.path()), (k, ls[k], lt[k])
