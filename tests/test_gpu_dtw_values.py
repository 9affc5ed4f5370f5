"""DTW over finite series whose squared differences or sums leave float32: the
costs are infinite, and scores and paths are still the oracle's."""

import numpy as np
import pytest

import oracle as O
import pyalign_amd as pa
from tests.test_gpu_parity import _dtw_oracle, rounded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("direction", ["minimize", "maximize"])
@pytest.mark.parametrize("scale", [1e13, 3e18, 3e19, 3e38])
def test_large_values(direction, scale):
    rng = np.random.default_rng(len(direction))
    pf = pa.series(direction=direction)
    data = [(rng.integers(-2, 3, size=(int(a), 2)).astype(np.float32), rng.integers(-2, 3, size=(int(b), 2)).astype(np.float32))
            for a, b in rng.integers(3, 90, size=(12, 2))]
    for x, y in data:  # (a few large values among small ones)
        x[rng.integers(0, len(x), 2)] = scale
        y[rng.integers(0, len(y))] = -scale / 2
    problems = [pf.new_problem(x, y) for x, y in data]
    lims = (rounded(max(len(x) for x, _ in data)), rounded(max(len(y) for _, y in data)))
    solutions = pa.ElasticSolver(codomain=pa.Solution).solve(problems)
    scores = pa.ElasticSolver(codomain=pa.Score).solve(problems)
    odir = O.MINIMIZE if direction == "minimize" else O.MAXIMIZE
    for k, (p, r, sc) in enumerate(zip(problems, solutions, scores)):
        with np.errstate(all="ignore"):
            ref = _dtw_oracle(p.matrix, odir, O.GOAL_ONE, lims)
        assert np.array_equal([r.score, sc], [ref.score, ref.score], equal_nan=True), k
        assert np.array_equal(np.asarray(r.path, dtype=np.int32), ref.path()), k
