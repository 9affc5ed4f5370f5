"""One-optimal results packed on the device (pa_pack_kernel): the alignment of
every path, in both index widths and for each workgroup size (a few, some
hundreds and thousands of problems), against the definition applied to the path
itself; results outlive the solver's next solve."""

import numpy as np
import pytest

import pyalign_amd as pa
from tests.test_gpu_parity import build_factory, random_bag

pytestmark = pytest.mark.gpu


def matched(path, ls, lt):
    s, t = np.full(ls, -1), np.full(lt, -1)
    for (a, b), (u, v) in zip(path[:-1], path[1:]):
        if u != a and v != b and a >= 0 and b >= 0:
            s[a], t[b] = b, a
    return s, t


@pytest.mark.parametrize("n", [1, 3, 300, 2100])
@pytest.mark.parametrize("limit", [64, 20000])  # int16 and int32 indices
@pytest.mark.parametrize("cls", [pa.GlobalSolver, pa.LocalSolver])
def test_alignments_of_paths(n, limit, cls):
    rng = np.random.default_rng(n + limit)
    _, pf = build_factory("binary", rng, "maximize")
    seqs, problems = random_bag(rng, pf, "ACGT", n, 0, 60)
    solver = cls(gap_cost=pa.AffineGapCost(2, 0.5), codomain=pa.Solution, max_len_s=limit, max_len_t=limit)
    first = solver.solve(problems)
    again = solver.solve(problems[::-1])[::-1]  # (reuses the solver's buffers)
    dtype = np.int16 if limit < 16000 else np.int32
    for (a, b), x, y in zip(seqs, first, again):
        if x.score is None:
            assert y.score is None and x.path is None and x.alignment is None
            continue
        assert x.score == y.score and np.array_equal(x.path, y.path) and x.path.dtype == dtype
        s, t = matched(x.path.tolist(), len(a), len(b))
        assert np.array_equal(x.alignment.s_to_t, s) and np.array_equal(x.alignment.t_to_s, t)
        assert x.alignment.s_to_t.dtype == dtype and x.alignment.score == x.score
        assert np.array_equal(y.alignment.s_to_t, s)
    only = cls(gap_cost=pa.AffineGapCost(2, 0.5), codomain=pa.Alignment, max_len_s=limit, max_len_t=limit)
    for x, al in zip(first, only.solve(problems)):
        if x.score is not None:
            assert al.score == x.score and np.array_equal(al.s_to_t, x.alignment.s_to_t)
            assert np.array_equal(al.t_to_s, x.alignment.t_to_s)
