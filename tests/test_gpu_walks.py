"""Trace walks against the oracle at the edges of their tiles: block sizes on
both sides of the matrix-instruction steps (1, 4, 6 and 16 states) and operator
lists shorter and longer than a walk's chunk of 16 operators."""

import dataclasses

import numpy as np
import pytest

from oracle import OracleChain
from w2dynamics_amd import problems as P
from w2dynamics_amd.ctqmc import CtqmcGpu
from test_gpu_parity import _compare

pytestmark = pytest.mark.gpu

# quantum numbers (blocks of a 2-orbital model), beta, TaudiffMax, moves
WALKS = {
    "nt_6states": ("Nt", 12.0, 3.0, 1500),
    "szt_6states_one_window": ("Szt", 10.0, -1.0, 1500),
    "one_block_16states": ("", 6.0, -1.0, 800),
    "blocks_to_4_one_window": ("Nt Szt", 14.0, -1.0, 1500),
}


@pytest.mark.parametrize("case", list(WALKS))
def test_walks_match_oracle(case):
    qn, beta, tdm, n = WALKS[case]
    prob = dataclasses.replace(P.kanamori_2orb(beta=beta, TaudiffMax=tdm), quantum_numbers=qn)
    print("walk", case, flush=True)
    gpu = CtqmcGpu.from_problem(prob, nchains=2, seed=515)
    gpu.set_taudiffmax(tdm)
    rec = gpu.moves_log(0, n)
    ora = OracleChain.from_problem(prob, 515)
    ora.set_taudiffmax(tdm)
    _compare(rec, ora.moves(n), case)
    assert np.max(rec["noper"]) > 8
    gpu.close()
