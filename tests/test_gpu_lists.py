"""Operator lists cut short so that more chains are resident, against full ones."""

import numpy as np
import pytest

from w2dynamics_amd import problems as P
from w2dynamics_amd.ctqmc import CtqmcError, CtqmcGpu

pytestmark = pytest.mark.gpu

DISCRETE = ("move", "kind", "outcome")


def _crowded(nf, pairs, t1):
    """pairs creator-annihilator pairs of every flavour, one after the other in (0, t1)."""
    fl = np.repeat(np.tile(np.arange(nf), pairs), 2)
    ca = np.tile([1, 2], nf * pairs)
    taus = (np.arange(fl.size) + 0.5) * (t1 / fl.size)
    return taus, fl // 2, fl % 2, ca


@pytest.mark.parametrize("crowd", [0, 42])
def test_short_lists_follow_full_lists(crowd):
    """A batch of 1024 chains holds lists of 488 operators where one chain holds
    800 (3 orbitals, capacity 384).  Both decide every move alike; a window of
    504 operators makes the batch return to full lists and go on.  Weights are
    sums of some 1e3 rounded logarithms: 1e3 x 2^-53 of their size."""
    prob = P.kanamori_3orb(beta=100.0, TaudiffMax=8.0)
    recs = []
    for nch in (1024, 1):
        print("lists", nch, "chains", crowd, flush=True)
        g = CtqmcGpu.from_problem(prob, nchains=nch, seed=77, capacity=384)
        g.set_taudiffmax(8.0)
        if crowd:
            cfg = _crowded(6, crowd, 15.0)
            # the outer block that the sequence leads back to: of the empty state
            for s in range(g.nsst):
                try:
                    g.set_config(0, *cfg, s)
                    break
                except CtqmcError:   # zero trace
                    continue
            assert g.get_config(0)["n"] == 12 * crowd
        recs.append(g.moves_log(0, 400))
        g.close()
    a, b = recs
    for k in a.dtype.names:
        if a[k].dtype.kind == "f":
            assert np.allclose(a[k], b[k], rtol=1e-12, atol=1e-12), k
        else:
            assert np.array_equal(a[k], b[k]), k
