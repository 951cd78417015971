"""The binning accumulator's batches of components against the oracle: fewer
components than a wavefront has lanes, a ragged last batch, a full one and one
component more; counts that fill the highest level."""

import numpy as np
import pytest

from oracle import OracleChain
from w2dynamics_amd import problems as P
from w2dynamics_amd.ctqmc import CtqmcGpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ntau,nmeas", [(5, 8), (129, 16), (256, 16), (257, 9), (1000, 4)])
def test_levels_match_oracle(ntau, nmeas):
    """Weights of the same moves differ by rounding: sums of some 1e3 terms,
    squared, hence 1e-9 of the largest variance."""
    prob = P.anderson_1orb(TaudiffMax=2.0, NCorr=20, Nmeas=nmeas, AccumGtau=2, Ntau=ntau)
    print("binning", ntau, nmeas, flush=True)
    gpu = CtqmcGpu.from_problem(prob, nchains=1, seed=33)
    ora = OracleChain.from_problem(prob, 33)
    for x in (gpu, ora):
        x.set_taudiffmax(2.0)
        x.warmup(400)
    gpu.measure(nmeas)
    ora.measure(nmeas, 20)
    a, b = gpu.gtau_blocks(0), ora.gtau_blocks()
    assert a.shape == b.shape
    fin = np.isfinite(b)
    assert np.array_equal(fin, np.isfinite(a))
    assert np.max(b[fin]) > 0
    assert np.allclose(a[fin], b[fin], rtol=1e-9, atol=1e-9 * np.max(b[fin]))
    gpu.close()
