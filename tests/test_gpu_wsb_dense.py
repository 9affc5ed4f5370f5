"""General gap costs over dense similarities given on the host, few (looked at
there) and many (looked at on the device): scores and paths against the oracle,
with and without a value whose folds depend on their order."""

import numpy as np
import pytest

import oracle as O
import pyalign_amd as pa
from pyalign_amd import algorithm
from tests.test_gpu_band import LOCS
from tests.test_gpu_wsb import STEPPY, oracle_gap

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("loc", list(LOCS))
@pytest.mark.parametrize("n", [3, 16])  # of 50 x 50: below and above 32,768 values
@pytest.mark.parametrize("value", [None, -0.0, np.inf, -np.inf, np.nan, 3e38])
def test_dense(loc, n, value):
    rng = np.random.default_rng(n + len(loc))
    S = rng.integers(-2, 3, (n, 50, 50)).astype(np.float32)
    S[S == 0] = 0.0
    if value is not None:
        S[n - 1, 20:, 20] = S[1, 0, 0] = value
    lens, off = np.full(n, 50, np.int32), np.arange(n) * 2500
    opts = dict(solver=algorithm.Type.ALIGNMENT, batch=True, direction=algorithm.Direction.MAXIMIZE, return_dup=False,
                codomain=pa.solve.Codomain(pa.Solution), locality=LOCS[loc][0], gap_cost=STEPPY)
    solver = algorithm.m16.create_solver(64, 64, algorithm.m16.create_options(opts))
    for _ in range(2):
        got = solver.solve_ragged("solution", "dense", lens, lens, dense=S.ravel(), dense_off=off)
        for k in (0, 1, n - 1):
            with np.errstate(all="ignore"):
                ref = O.OracleResult(O.make_config(locality=LOCS[loc][1], gap=oracle_gap(STEPPY, (64, 64)),
                                                   goal=O.GOAL_ONE, lim_s=64, lim_t=64), S[k])
            if not ref.has_seed:
                assert got[k].score is None, k
                continue
            assert np.array_equal(np.float32(got[k].score), ref.score, equal_nan=True), k
            assert np.array_equal(np.asarray(got[k].path, np.int32), ref.path()), k
