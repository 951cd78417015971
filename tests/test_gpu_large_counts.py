"""Move counts beyond 32 bits: window slides further apart than any 32-bit
number of moves, against the oracle."""

import pytest

from oracle import OracleChain
from test_gpu_parity import _compare
from w2dynamics_amd import problems as P
from w2dynamics_amd.ctqmc import CtqmcGpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slide", [2**31 - 1, 2**31, 2**32 + 3])
def test_rare_slides_match_oracle(slide):
    """Four windows: NSlide = NCorr / 4, so that the window stays where it is."""
    prob = P.anderson_1orb(TaudiffMax=2.0, NCorr=4 * slide)
    print("slide", slide, flush=True)
    gpu = CtqmcGpu.from_problem(prob, nchains=1, seed=31)
    gpu.set_taudiffmax(2.0)
    rec = gpu.moves_log(0, 400)
    ora = OracleChain.from_problem(prob, 31)
    ora.set_taudiffmax(2.0)
    _compare(rec, ora.moves(400), "slide %d" % slide)
    assert rec["noper"].max() > 0
    gpu.close()
