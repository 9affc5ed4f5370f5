"""Tables that differ in the sign of a zero only, one after the other on one
solver: every score bit for bit the oracle's (an earlier table's -0 must not
stand in for +0, nor the other way round)."""

import numpy as np
import pytest
import torch

import oracle as O
import pyalign_amd as pa
from tests.test_gpu_band import LOCS, make_solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["score", "solution"])
@pytest.mark.parametrize("gap", [("affine", 1, 1), ("linear", 2)], ids=str)
def test_sign_of_zero(kind, gap):
    solver = make_solver("global", gap, "maximize", pa.Score if kind == "score" else pa.Solution, 8, 8)
    one, codes, off = np.ones(3, np.int32), np.array([0, 1, 0], np.uint8), np.arange(3)
    streams = [None, torch.cuda.Stream().cuda_stream]
    for q, zero in enumerate([0.0, -0.0, 0.0, 0.0, -0.0, -0.0, 0.0]):
        solver.set_stream(streams[q // 2 % 2])
        table = np.full((2, 2), zero, np.float32)
        got = solver.solve_ragged(kind, "indexed", one, one, codes_s=codes, codes_t=codes, off_s=off, off_t=off,
                                  table=table)
        for k in range(3):
            ref = O.OracleResult(O.make_config(locality=LOCS["global"][1], gap=gap,
                                               goal=O.GOAL_SCORE if kind == "score" else O.GOAL_ONE, lim_s=8,
                                               lim_t=8), table[:1, :1])
            score = got[k] if kind == "score" else got[k].score
            assert np.float32(score).tobytes() == ref.score.tobytes(), (q, k)
