"""The score kernel's local maximum over a table takes any table without NaN, a
-0 among them: scores against the strict folds, which a NaN in an entry that no
sequence uses selects, and a sample against the oracle."""

import numpy as np
import pytest

import oracle as O
import pyalign_amd as pa
from tests.test_gpu_band import LOCS, make_solver, sym_table
from tests.test_gpu_score_kernel import GAPS, bag

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gap", GAPS, ids=str)
@pytest.mark.parametrize("zero", [0.0, -0.0])
@pytest.mark.parametrize("n", [200, 4000])
def test_local_maximum(gap, zero, n):
    rng = np.random.default_rng(n)
    ls, lt, cs, ct, os_, ot = bag(rng, n, 5)
    table = sym_table(rng, 6, -3, 4)
    table[table == 0] = zero
    table[0, 1] = -np.inf
    strict = table.copy()
    strict[5, 5] = np.nan
    got, want = (make_solver("local", gap, "maximize", pa.Score, 1024, 2048).solve_ragged(
        "score", "indexed", ls, lt, codes_s=cs, codes_t=ct, off_s=os_, off_t=ot, table=t) for t in (table, strict))
    assert np.array_equal(np.asarray(got, np.float32).view(np.uint32), np.asarray(want, np.float32).view(np.uint32))
    for k in range(0, n, n // 40):
        S = table[cs[os_[k]:os_[k] + ls[k]]][:, ct[ot[k]:ot[k] + lt[k]]]
        ref = O.OracleResult(O.make_config(locality=LOCS["local"][1], gap=gap, goal=O.GOAL_SCORE, lim_s=1024,
                                           lim_t=2048), S)
        assert np.float32(got[k]).tobytes() == ref.score.tobytes(), (k, ls[k], lt[k])
