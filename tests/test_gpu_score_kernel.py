"""Alignments over tables and binary symbols with max / min folds: the score
kernel (every locality, direction and gap model) and the max-folding traceback
kernel.  Bit for bit against the strict folds, which a -0 in a table entry that
no sequence uses selects, and against the oracle.
"""

import numpy as np
import pytest

import oracle as O
import pyalign_amd as pa
from tests.test_gpu_band import LOCS, dense_of, lengths, make_solver, ragged_codes, sym_table

pytestmark = pytest.mark.gpu

GAPS = [("affine", 5, 1), ("affine", 3, 0), ("linear", 2)]


def bag(rng, n, K):
    """Tiny to tall problems: one lane each, several strips, odd lengths."""
    ls, lt = lengths(rng, n, 1, 40, 1, 40)
    for k, (a, b) in enumerate([(700, 900), (1, 600), (600, 1), (513, 300), (512, 70), (97, 1100), (0, 5), (5, 0)]):
        ls[k], lt[k] = a, b
    cs, ct, os_, ot = ragged_codes(rng, ls, lt, K)
    return ls, lt, cs, ct, os_, ot


@pytest.mark.parametrize("loc", list(LOCS))
@pytest.mark.parametrize("gap", GAPS, ids=str)
@pytest.mark.parametrize("direction", ["maximize", "minimize"])
@pytest.mark.parametrize("n", [200, 4000])
def test_table_folds(loc, gap, direction, n):
    rng = np.random.default_rng(n + 10 * len(loc) + len(direction))
    ls, lt, cs, ct, os_, ot = bag(rng, n, 5)
    ls[8:n // 2] += 100  # (their codes are read where they are: any symbols)
    os_[8:] = rng.integers(0, len(cs) - 200, n - 8)
    ot[8:] = rng.integers(0, len(ct) - 200, n - 8)
    table = sym_table(rng, 6, -3, 4)
    table[table == 0] = 0.0  # (no -0 left by the symmetrisation)
    if direction == "minimize":
        table = np.where(table == 0, 0.0, -table).astype(np.float32)
    table[0, 1] = -np.inf if direction == "maximize" else np.inf  # (a pair that never matches)
    strict = table.copy()
    strict[5, 5] = -0.0
    payload = dict(codes_s=cs, codes_t=ct, off_s=os_, off_t=ot)
    for codomain, kind in ((pa.Score, "score"), (pa.Solution, "solution")):
        a, b = (make_solver(loc, gap, direction, codomain, 1024, 2048).solve_ragged(kind, "indexed", ls, lt, table=t,
                                                                                  **payload) for t in (table, strict))
        if kind == "score":
            assert np.array_equal(np.asarray(a, np.float32).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))
            continue
        for k in range(n):
            assert (a[k].score is None) == (b[k].score is None), k
            if a[k].score is not None:
                assert np.float32(a[k].score).tobytes() == np.float32(b[k].score).tobytes(), k
                assert np.array_equal(a[k].path, b[k].path), (k, ls[k], lt[k])


@pytest.mark.parametrize("loc", list(LOCS))
@pytest.mark.parametrize("direction", ["maximize", "minimize"])
@pytest.mark.parametrize("odd", [None, "worst", "-0", "inf", "nan"])
def test_dense_folds(loc, direction, odd):
    """Dense similarities: codes from signs, and strict folds again for the
    groups that meet a value max / min folds cannot take."""
    rng = np.random.default_rng(3 + len(loc))
    n = 60
    ls, lt = lengths(rng, n, 1, 90, 8, 90)
    ls[:3], lt[:3] = (600, 513, 64), (40, 33, 500)
    flat = rng.integers(-2, 3, int((ls.astype(np.int64) * lt).sum())).astype(np.float32)
    flat[flat == 0] = 0.0
    off = np.concatenate([[0], np.cumsum(ls.astype(np.int64) * lt)[:-1]])
    if odd:
        bad = {"worst": -np.inf if direction == "maximize" else np.inf, "-0": -0.0,
               "inf": np.inf if direction == "maximize" else -np.inf, "nan": np.nan}[odd]
        for k in (0, 5, 17):
            flat[off[k] + rng.integers(0, ls[k] * lt[k], 3)] = bad
        flat[off[9]] = bad  # the first cell: -0 beside the border's -0
    odir = O.MAXIMIZE if direction == "maximize" else O.MINIMIZE
    for gap in GAPS:
        got = make_solver(loc, gap, direction, pa.Solution, 1024, 1024).solve_ragged("solution", "dense", ls, lt,
                                                                                   dense=flat, dense_off=off)
        for k in range(n):
            S = flat[off[k]:off[k] + ls[k] * lt[k]].reshape(ls[k], lt[k])
            ref = O.OracleResult(O.make_config(locality=LOCS[loc][1], direction=odir, gap=gap, goal=O.GOAL_ONE,
                                               lim_s=1024, lim_t=1024), S)
            if not ref.has_seed:
                assert got[k].score is None, k
                continue
            assert np.float32(got[k].score).tobytes() == ref.score.tobytes(), (k, gap)
            assert np.array_equal(np.asarray(got[k].path, np.int32), ref.path()), (k, gap)


@pytest.mark.parametrize("loc", list(LOCS))
@pytest.mark.parametrize("gap", GAPS, ids=str)
@pytest.mark.parametrize("eq,ne,direction", [(2.0, -1.0, "maximize"), (1.0, 0.0, "maximize"), (1.0, 0.5, "maximize"),
                                             (-2.0, 1.0, "minimize"), (0.0, 1.0, "minimize")])
def test_binary_folds(loc, gap, eq, ne, direction):
    rng = np.random.default_rng(7 + len(loc))
    ls, lt, cs, ct, os_, ot = bag(rng, 60, 3)
    cs, ct = cs.astype(np.uint32), ct.astype(np.uint32)
    cs[cs == 2] = 0xffffffff  # (code values are compared, whatever they are)
    ct[ct == 2] = 0xffffffff
    odir = O.MAXIMIZE if direction == "maximize" else O.MINIMIZE
    for codomain, kind, goal in ((pa.Score, "score", O.GOAL_SCORE), (pa.Solution, "solution", O.GOAL_ONE)):
        got = make_solver(loc, gap, direction, codomain, 1024, 2048).solve_ragged(
            kind, "binary", ls, lt, codes_s=cs, codes_t=ct, off_s=os_, off_t=ot, eq=eq, ne=ne)
        for k in range(len(ls)):
            S = dense_of("binary", k, cs, ct, os_, ot, ls, lt, None, eq, ne)
            ref = O.OracleResult(O.make_config(locality=LOCS[loc][1], direction=odir, gap=gap, goal=goal, lim_s=1024,
                                               lim_t=2048), S)
            if kind == "score":
                assert np.float32(got[k]).tobytes() == ref.score.tobytes(), (k, ls[k], lt[k])
            elif not ref.has_seed:
                assert got[k].score is None
            else:
                assert np.float32(got[k].score).tobytes() == ref.score.tobytes(), (k, ls[k], lt[k])
                assert np.array_equal(np.asarray(got[k].path, np.int32), ref.path()), (k, ls[k], lt[k])
