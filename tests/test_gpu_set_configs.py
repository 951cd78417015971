"""Configurations of a batch set in one call against one call per chain."""

import numpy as np
import pytest

from w2dynamics_amd import problems as P
from w2dynamics_amd.ctqmc import CtqmcError, CtqmcGpu, _p

pytestmark = pytest.mark.gpu

KEYS = ("trace_log", "trace_sign", "det_log", "det_sign", "cfgsign")


def _set(gpu, cfgs):
    off = np.concatenate([[0], np.cumsum([c["n"] for c in cfgs])]).astype(np.int64)
    cat = lambda k, dt: np.ascontiguousarray(np.concatenate([c[k] for c in cfgs]), dt)   # noqa: E731
    tau, orb, spin, ca = cat("taus", np.float64), cat("orbs", np.int32), cat("spins", np.int32), cat("cas", np.int32)
    outer = np.array([c["outer_sst"] for c in cfgs], np.int32)
    w = np.zeros((len(cfgs), 5))
    st = gpu.lib.w2d_ctqmc_set_configs(gpu.h, len(cfgs), _p(off), _p(tau), _p(orb), _p(spin), _p(ca), _p(outer), _p(w))
    return st, w


@pytest.mark.parametrize("build,kw,nch", [(P.anderson_1orb, dict(beta=10.0), 7),
                                          (P.kanamori_2orb, dict(beta=16.0), 5),
                                          (P.kanamori_3orb, dict(beta=6.0), 3)])
def test_batch_equals_single_calls(build, kw, nch):
    """Same weights as set_config chain by chain, empty configurations among
    them, in a handle whose capacity has to grow; a configuration that is refused
    stops the batch behind the ones before it."""
    prob = build(TaudiffMax=-1.0, **kw)
    print("set_configs", prob.label, nch, flush=True)
    a = CtqmcGpu.from_problem(prob, nchains=nch, seed=21)
    empty = a.get_config(0)
    a.warmup(1500)
    cfgs = [a.get_config(c) for c in range(nch)]
    cfgs[1] = dict(empty, outer_sst=cfgs[1]["outer_sst"])
    assert max(c["n"] for c in cfgs) > 4
    ref = np.array([[a.set_config(c, *[x[k] for k in ("taus", "orbs", "spins", "cas", "outer_sst")])[k2]
                     for k2 in KEYS] for c, x in enumerate(cfgs)])
    b = CtqmcGpu.from_problem(prob, nchains=nch, seed=22, capacity=256)
    st, w = _set(b, cfgs)
    assert st == 0
    assert np.array_equal(w, ref)
    for c in range(nch):
        g = b.get_config(c)
        assert all(np.array_equal(g[k], cfgs[c][k]) for k in ("taus", "orbs", "spins", "cas", "outer_sst")), c
    # refused: not sorted; chains before it are set, the ones behind keep theirs
    bad = dict(cfgs[2], taus=cfgs[2]["taus"][::-1].copy())
    fresh = CtqmcGpu.from_problem(prob, nchains=nch, seed=23)
    st, _ = _set(fresh, cfgs[:2] + [bad] + cfgs[3:])
    assert st == 1
    assert fresh.get_config(0)["n"] == cfgs[0]["n"] and fresh.get_config(2)["n"] == 0
    with pytest.raises(CtqmcError):
        fresh.set_config(2, *[bad[k] for k in ("taus", "orbs", "spins", "cas", "outer_sst")])
    for g in (a, b, fresh):
        g.close()
