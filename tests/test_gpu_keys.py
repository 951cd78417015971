"""Quantum-number look-ups of proposals against the oracle's walks: windows that
hold no operator, more operators between a pair than a wavefront has lanes, and
blocks on both sides of 4 states."""

import numpy as np
import pytest

from oracle import OracleChain
from w2dynamics_amd import problems as P
from w2dynamics_amd.ctqmc import CtqmcGpu
from test_gpu_parity import _compare

pytestmark = pytest.mark.gpu

# model, beta, TaudiffMax, moves, operators reached
RUNS = {
    "empty_windows": (P.anderson_1orb, 4.0, 0.5, 4000, 2),
    "2orb_beyond_a_wave": (P.kanamori_2orb, 60.0, -1.0, 16000, 70),
    "3orb_beyond_a_wave": (P.kanamori_3orb, 40.0, -1.0, 8000, 66),
    "3orb_windows": (P.kanamori_3orb, 12.0, 2.0, 1200, 10),
}


@pytest.mark.parametrize("run", list(RUNS))
def test_refused_proposals_match_oracle(run):
    model, beta, tdm, n, nops = RUNS[run]
    prob = model(beta=beta, TaudiffMax=tdm)
    print("keys", run, flush=True)
    gpu = CtqmcGpu.from_problem(prob, nchains=2, seed=909)
    gpu.set_taudiffmax(tdm)
    rec = gpu.moves_log(1, n)
    ora = OracleChain.from_problem(prob, 910)
    ora.set_taudiffmax(tdm)
    _compare(rec, ora.moves(n), run)
    assert np.max(rec["noper"]) >= nops
    gpu.close()
