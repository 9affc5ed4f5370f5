"""A captured launch sequence is replayed only for the same arguments: one long
pair solved again and again on one solver with other symbol scores and gap
costs between, every score and path against the oracle."""

import numpy as np
import pytest

import oracle as O
import pyalign_amd as pa
from tests.test_gpu_band import LOCS, dense_of, make_solver, ragged_codes, sym_table

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("change", ["scores", "gap", "form"])
def test_long_pair_after_a_change(change):
    rng = np.random.default_rng(len(change))
    ls, lt = np.array([1024], np.int32), np.array([1500], np.int32)
    cs, ct, os_, ot = ragged_codes(rng, ls, lt, 4)
    table = sym_table(rng, 4)
    wide = (cs.astype(np.uint32), ct.astype(np.uint32))
    solver = make_solver("global", ("affine", 5, 1), "maximize", pa.Solution, 1024, 2048)
    first, second = ("binary", (2.0, -1.0), 5), {"scores": ("binary", (1.0, -3.0), 5), "gap": ("binary", (2.0, -1.0), 2),
                                                 "form": ("indexed", None, 5)}[change]
    for form, scores, opened in (first, second, second, first, first, first, second):
        solver.set_gap_cost(pa.AffineGapCost(opened, 1))
        if form == "binary":
            got = solver.solve_ragged("solution", form, ls, lt, codes_s=wide[0], codes_t=wide[1], off_s=os_, off_t=ot,
                                      eq=scores[0], ne=scores[1])
        else:
            got = solver.solve_ragged("solution", form, ls, lt, codes_s=cs, codes_t=ct, off_s=os_, off_t=ot, table=table)
        assert solver.last_schedule()[:2] == (0, 1)  # long mode and no other launch
        S = dense_of(form, 0, cs, ct, os_, ot, ls, lt, table, *(scores or (0, 0)))
        ref = O.OracleResult(O.make_config(locality=LOCS["global"][1], gap=("affine", opened, 1), goal=O.GOAL_ONE,
                                           lim_s=1024, lim_t=2048), S)
        assert np.float32(got[0].score).tobytes() == ref.score.tobytes(), (form, scores, opened)
        assert np.array_equal(np.asarray(got[0].path, dtype=np.int32), ref.path()), (form, scores, opened)
