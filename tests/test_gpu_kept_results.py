"""What Solutions and Alignments keep alive: never the native result (its
pinned buffer goes back to the solver's pool as the solve ends), and an
Alignment only the maps of its bag, not the paths nor the problems' data."""

import gc
import weakref

import numpy as np
import pytest

import pyalign_amd as pa
from pyalign_amd import algorithm
from tests.test_gpu_parity import build_factory, random_bag

pytestmark = pytest.mark.gpu


def solved(n, times):
    rng = np.random.default_rng(n)
    _, pf = build_factory("binary", rng, "maximize")
    seqs, problems = random_bag(rng, pf, "ACGT", n, 1, 40)
    solver = pa.GlobalSolver(gap_cost=pa.AffineGapCost(2, 0.5), codomain=pa.Solution)
    kept = [solver.solve(problems if n > 1 else problems[0]) for _ in range(times)]
    return seqs, kept if n > 1 else [[x] for x in kept]


@pytest.mark.parametrize("n", [1, 40])
def test_results_are_freed_at_once(n, monkeypatch):
    made = []

    class Watched(algorithm._Result):
        def __init__(self, *args):
            super().__init__(*args)
            made.append(weakref.ref(self))

    monkeypatch.setattr(algorithm, "_Result", Watched)
    seqs, kept = solved(n, 3)
    gc.collect()
    assert len(made) >= 3 and not any(r() for r in made)
    for (a, b), x in zip(seqs, kept[0]):  # (matrices are still made from the problem's data)
        assert x.values.shape[-2:] == (len(a) + 1, len(b) + 1)


def test_an_alignment_keeps_the_maps_only():
    seqs, (solutions,) = solved(50, 1)
    want = [(x.score, x.path.copy(), x.alignment.s_to_t.copy()) for x in solutions]
    alignments = [x.alignment for x in solutions]
    core = [x._solution.alignment for x in solutions]  # (the core solver's own)
    del solutions
    gc.collect()
    assert not [x for x in gc.get_objects() if type(x) in (algorithm._Solved, algorithm._BagSolution)]
    for al, own, (score, path, s_to_t) in zip(alignments, core, want):
        assert al.score == score == own.score and al.s_to_t is al.s_to_t and al.t_to_s is al.t_to_s
        assert np.array_equal(al.s_to_t, s_to_t) and np.array_equal(own.s_to_t, s_to_t)
        assert np.array_equal(al.t_to_s, own.t_to_s)
        assert [tuple(e) for e in al.edges] == [(i, j) for i, j in enumerate(s_to_t) if j >= 0]
