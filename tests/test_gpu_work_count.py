"""The count of arithmetic that a chain reports, against the formula, where only
global moves are made."""

import numpy as np
import pytest

from w2dynamics_amd import problems as P
from w2dynamics_amd.ctqmc import CtqmcGpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 5, 20])
def test_global_moves_count_what_they_do(k):
    """One-state blocks, k pairs in both flavours.  A global move that quantum
    numbers allow factorises each flavour's matrix once, 2/3 k^3, and walks the
    configuration once, 3 operations an operator; an accepted one inverts the
    matrices, 2 k^3.  The one measurement adds k^2 (5 NLegMax + 4) a flavour."""
    beta, nmoves, nleg = 10.0, 200, 10
    prob = P.anderson_1orb(beta=beta, TaudiffMax=-1.0, NCorr=nmoves, NLegMax=nleg, MeasDensityMatrix=0,
                           PercentageGlobalMove=1.0, PercentageTauShiftMove=0.0)
    t = (np.arange(4 * k) + 0.5) * (beta / (4 * k))
    spins = np.tile([0, 0, 1, 1], k)
    cas = np.tile([1, 2, 1, 2], k)
    print("work", k, flush=True)
    g = CtqmcGpu.from_problem(prob, nchains=1, seed=81)
    m = g.model()
    outer = next(q for q, (o, n) in enumerate(zip(m["offsets"], m["sizes"])) if 0 in m["states"][o:o + n])
    g.set_config(0, t, np.zeros(4 * k, int), spins, cas, outer)
    g.measure(1)
    sc = g.accumulators()["scalars"][0]
    acc, tried, moves, qn, flops = sc[6], sc[7], sc[10], sc[11], sc[12]
    assert moves == tried == nmoves
    expect = (tried - qn) * (2 * (2 / 3) * k**3 + 3 * 4 * k) + acc * 2 * 2 * k**3 + 2 * k**2 * (5 * nleg + 4)
    assert acc > 0 and np.isclose(flops, expect, rtol=1e-12), (flops, expect, acc, qn)
    g.close()
