"""Chains that start from a stored configuration of zero weight, against the oracle."""

import dataclasses

import numpy as np
import pytest

from oracle import OracleChain
from test_gpu_parity import _compare
from w2dynamics_amd import problems as P
from w2dynamics_amd.ctqmc import CtqmcGpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [5, 6, 7])
def test_sign_returns_with_the_weight(seed):
    """Two creators of one flavour in a row: allowed by the electron number, a
    zero of the trace (exactly, all matrix elements being 0 or 1).  The first
    accepted move to a nonzero weight has its sign."""
    beta = 6.0
    prob = dataclasses.replace(P.anderson_1orb(beta=beta, TaudiffMax=-1.0), quantum_numbers="Nt")
    cfg = (np.array([0.15, 0.35, 0.6, 0.85]) * beta, np.zeros(4, int), np.zeros(4, int), np.array([1, 1, 2, 2]))
    print("zero weight", seed, flush=True)
    gpu = CtqmcGpu.from_problem(prob, nchains=1, seed=seed)
    ora = OracleChain.from_problem(prob, seed)
    m = gpu.model()
    outer = next(q for q, (o, n) in enumerate(zip(m["offsets"], m["sizes"])) if 0 in m["states"][o:o + n])
    assert gpu.set_config(0, *cfg, outer)["trace_sign"] == 0.0
    ora.set_config(*cfg, outer)
    rec = gpu.moves_log(0, 300)
    ref = ora.moves(300)
    assert ref["cfgsign"][-1] != 0.0
    _compare(rec, ref, "zero weight")
    gpu.close()
