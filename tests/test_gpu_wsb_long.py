"""General gap costs of one long pair: more to push on along an anti-diagonal
than a launch has workgroups for, so that each takes several turns; score and
path against the oracle."""

import numpy as np
import pytest

import oracle as O
import pyalign_amd as pa
from tests.test_gpu_parity import SOLVERS, build_factory, dense
from tests.test_gpu_wsb import oracle_gap

pytestmark = pytest.mark.gpu

LONG = 66000  # 4,125 blocks


@pytest.mark.parametrize("loc,lims", [("global", (1, LONG)), ("semiglobal", (LONG, 1))])
def test_turns(loc, lims):
    rng = np.random.default_rng(5)
    alphabet, pf = build_factory("binary", rng, "maximize")
    problem = pf.new_problem(*("".join(rng.choice(list(alphabet), k)) for k in lims))
    cls, oloc = SOLVERS[loc]
    gap = pa.LogarithmicGapCost(2, 0.7)
    got = cls(gap_cost=gap, codomain=pa.Solution).solve([problem, pf.new_problem("A", "A")])[0]
    ref = O.OracleResult(O.make_config(locality=oloc, gap=oracle_gap(gap, lims), goal=O.GOAL_ONE, index_bits=32,
                                       lim_s=lims[0], lim_t=lims[1]), dense(problem))
    assert np.float32(got.score).tobytes() == ref.score.tobytes()
    assert np.array_equal(np.asarray(got.path, dtype=np.int32), ref.path())
