"""General gap costs in blocks of 16 x 16 cells (scores and one optimal path)
against the oracle, bit for bit: block edges and remainders, the three ways
blocks share a workgroup (four problems, neighbours of one problem, carried
sums), and values whose folds depend on the order (served by the cell-by-cell
kernel).
"""

import zlib

import numpy as np
import pytest

import oracle as O
import pyalign_amd as pa
from tests.test_gpu_parity import SOLVERS, build_factory, dense, rounded
from tests.test_gpu_wsb import STEPPY, oracle_gap

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 15, 16, 17, 31, 32, 33, 47, 49]
# (lengths of s, lengths of t): many problems (workgroups take four), a few
# short ones (four neighbouring blocks of one), long ones (carried sums)
BAGS = {"many": ([EDGES[k % 10] for k in range(40)], [EDGES[(k // 4 + 3 * k) % 10] for k in range(40)]),
        "few": ([100, 65, 16], [33, 112, 150]),
        "one": ([64], [129]),
        "carried": ([400, 17, 385, 1], [37, 380, 401, 500])}


def check(solver, problems, oloc, odir, gap, lims):
    got = solver.solve(problems)
    for p, g in zip(problems, got):
        ref = O.OracleResult(O.make_config(locality=oloc, direction=odir, gap=oracle_gap(gap, lims), goal=O.GOAL_ONE,
                                           lim_s=lims[0], lim_t=lims[1]), dense(p))
        if not ref.has_seed:
            assert g.score is None and g.path is None
            continue
        assert np.float32(g.score).tobytes() == ref.score.tobytes(), p.shape
        assert np.array_equal(np.asarray(g.path, dtype=np.int32), ref.path()), p.shape


def problems_of(rng, form, direction, bag):
    alphabet, pf = build_factory(form, rng, direction)
    letters = list(alphabet)
    out = []
    for a, b in zip(*BAGS[bag]):
        out.append(pf.new_problem("".join(rng.choice(letters, a)), "".join(rng.choice(letters, b))))
    lims = (rounded(max(BAGS[bag][0])), rounded(max(BAGS[bag][1])))
    return out, lims


@pytest.mark.parametrize("loc", list(SOLVERS))
@pytest.mark.parametrize("bag", list(BAGS))
@pytest.mark.parametrize("direction,form", [("maximize", "alphabetic"), ("minimize", "binary"), ("maximize", "general")])
def test_blocks(loc, bag, direction, form):
    rng = np.random.default_rng(zlib.crc32(repr((loc, bag, direction, form)).encode()))
    problems, lims = problems_of(rng, form, direction, bag)
    cls, oloc = SOLVERS[loc]
    odir = O.MAXIMIZE if direction == "maximize" else O.MINIMIZE
    for gap in (pa.LogarithmicGapCost(2, 0.7), STEPPY):
        solver = cls(gap_cost=gap, codomain=pa.Solution)
        if len(problems) > 1:
            check(solver, problems, oloc, odir, gap, lims)
        else:
            got = solver.solve(problems[0])
            check(type("One", (), {"solve": lambda self, p: [got]})(), problems, oloc, odir, gap, lims)


@pytest.mark.parametrize("loc", list(SOLVERS))
@pytest.mark.parametrize("values", ["negative zero", "free gap", "infinite cost", "infinite similarity"])
def test_order_dependent_values(loc, values):
    rng = np.random.default_rng(zlib.crc32(repr((loc, values)).encode()))
    t = rng.integers(-2, 3, size=(4, 4)).astype(np.float32)
    gap = pa.UserFuncGapCost(lambda k: [0, 2, 3, 3][min(k, 3)])
    if values == "negative zero":
        t[t == 0] = -0.0
        t[1, 2] = -0.0
    elif values == "free gap":  # w(1) = 0: border cells and costs of -0
        gap = pa.UserFuncGapCost(lambda k: 0 if k < 2 else 1)
    elif values == "infinite cost":
        gap = pa.UserFuncGapCost(lambda k: np.inf if k > 5 else float(k))
    else:
        t[0, 0] = np.inf
        t[2, 3] = -np.inf
    lookup = {(x, y): t[i, j] for i, x in enumerate("ACGT") for j, y in enumerate("ACGT")}
    pf = pa.alphabetic("ACGT", lambda x, y: lookup[(x, y)])
    problems = [pf.new_problem("".join(rng.choice(list("ACGT"), rng.integers(1, 40))),
                               "".join(rng.choice(list("ACGT"), rng.integers(1, 40)))) for _ in range(6)]
    lims = (rounded(max(p.shape[0] for p in problems)), rounded(max(p.shape[1] for p in problems)))
    cls, oloc = SOLVERS[loc]
    check(cls(gap_cost=gap, codomain=pa.Solution), problems, oloc, O.MAXIMIZE, gap, lims)
