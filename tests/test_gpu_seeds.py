"""Random streams seeded on the device against the oracle's: the edges of the
32-bit seed, and a chain whose seed wraps around."""

import numpy as np
import pytest

from oracle import OracleChain
from w2dynamics_amd import problems as P
from w2dynamics_amd.ctqmc import CtqmcGpu
from test_gpu_parity import _compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed,chain", [(0, 0), (2**32 - 1, 0), (2**32 - 1, 1), (5, 299)])
def test_streams_match_oracle(seed, chain):
    prob = P.anderson_1orb(TaudiffMax=2.0)
    print("seed", seed, "chain", chain, flush=True)
    gpu = CtqmcGpu.from_problem(prob, nchains=chain + 1, seed=seed)
    gpu.set_taudiffmax(2.0)
    rec = gpu.moves_log(chain, 800)
    ora = OracleChain.from_problem(prob, (seed + chain) % 2**32)
    ora.set_taudiffmax(2.0)
    _compare(rec, ora.moves(800), "seed %d chain %d" % (seed, chain))
    assert np.max(rec["noper"]) > 0
    gpu.close()
