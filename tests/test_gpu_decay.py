"""Cached states that decay at every operator, against the oracle."""

import dataclasses

import numpy as np
import pytest

from oracle import OracleChain
from test_gpu_parity import FIELDS
from w2dynamics_amd import problems as P
from w2dynamics_amd.ctqmc import CtqmcGpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("norb,tdm,scale,seed", [(2, 8.0, 1.0, 103), (2, 8.0, 1.0, 104), (2, 8.0, 1.0, 107),
                                                 (2, 8.0, 1.0, 113), (2, 8.0, 1.0, 119), (2, 8.0, 1.0, 250),
                                                 (3, 3.0, 0.45, 120)])
def test_decaying_states_match_oracle(norb, tdm, scale, seed):
    """Density interaction (matrix elements are 0 or 1: no rounding to hide
    behind) and a crystal field of 50: the highest orbital stays occupied while
    the lowest one empties and fills, so that the state of the chain is the
    highest of its block at nearly every operator and shrinks by up to exp(-95)
    beside the block's lowest.  Prefix kets and suffix bras of the window grow by
    a few operators at a time.  Weights are sums of about 100 rounded logarithms:
    100 x 2^-53 of their size."""
    cf = np.array([0.0, 50.0, 40.0])[:norb]
    d1, d2 = 1.9 * scale, 0.95 * scale
    ops, t = [(1.0, 1, 1, 1)], 1.0 + d1
    for _ in range(24):
        ops += [(t, 0, 0, 2), (t + d2, 0, 0, 1)]
        t = t + d2 + d1
    ops.append((t, 1, 1, 2))
    build = {2: P.kanamori_2orb, 3: P.kanamori_3orb}[norb]
    prob = dataclasses.replace(build(beta=t + 1.0, TaudiffMax=tdm), umatrix=P.u_kanamori(norb, 4.0, 2.0, 0.0),
                               muimp=P.solver_muimp(norb, 3.5, cf))
    cfg = [np.array(x) for x in zip(*ops)]
    print("decay", norb, tdm, scale, seed, flush=True)
    gpu = CtqmcGpu.from_problem(prob, nchains=1, seed=seed)
    ora = OracleChain.from_problem(prob, seed)
    for x in (gpu, ora):
        x.set_taudiffmax(tdm)
    m = gpu.model()
    outer = next(q for q, (o, n) in enumerate(zip(m["offsets"], m["sizes"])) if 3 in m["states"][o:o + n])
    gpu.set_config(0, *cfg, outer)
    ora.set_config(*cfg, outer)
    rec, ref = gpu.moves_log(0, 40), ora.moves(40)
    for f in FIELDS:
        assert np.array_equal(rec[f], ref[f]), f
    for f in ("trace_log", "det_log"):
        assert np.allclose(rec[f], ref[f], rtol=1e-12, atol=1e-12), f
    gpu.close()
