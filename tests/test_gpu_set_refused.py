"""A batch of configurations with one that the device refuses, against one call
per chain: the chains behind it keep their configurations."""

import dataclasses

import numpy as np
import pytest

from w2dynamics_amd import problems as P
from w2dynamics_amd.ctqmc import CtqmcError, CtqmcGpu

pytestmark = pytest.mark.gpu

ORDER = ("taus", "orbs", "spins", "cas", "outer_sst")


def _deaf(prob):
    """The same problem with the hybridisation of the last flavour at zero: its
    matrix is singular."""
    f = np.array(prob.ftau)
    f[-1, 1, -1, 1] = 0.0
    return dataclasses.replace(prob, ftau=f)


def _pair(beta, orb, spin, ca):
    return dict(taus=np.array([0.25, 0.5]) * beta, orbs=np.full(2, orb), spins=np.full(2, spin), cas=np.array(ca))


# model, error of the refused configuration, flavour of its pair
CASES = {
    "1state_trace": (lambda: P.anderson_1orb(beta=10.0, TaudiffMax=-1.0), 5),
    "4state_trace": (lambda: P.kanamori_2orb(beta=16.0, TaudiffMax=-1.0), 5),
    "9state_trace": (lambda: P.kanamori_3orb(beta=6.0, TaudiffMax=-1.0), 5),
    "1state_singular": (lambda: _deaf(P.anderson_1orb(beta=10.0, TaudiffMax=-1.0)), 4),
    "4state_singular": (lambda: _deaf(P.kanamori_2orb(beta=16.0, TaudiffMax=-1.0)), 4),
    "9state_singular": (lambda: _deaf(P.kanamori_3orb(beta=6.0, TaudiffMax=-1.0)), 4),
}


def _outer(g, bits):
    """superstate that holds the occupation state"""
    m = g.model()
    return next(q for q, (o, n) in enumerate(zip(m["offsets"], m["sizes"])) if bits in m["states"][o:o + n])


@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("where", [0, 2, 4])
def test_chains_behind_a_refused_one_keep_theirs(case, where, tmp_path):
    build, code = CASES[case]
    prob = build()
    nb, nch = prob.nbands, 5
    print("refused", case, where, flush=True)
    src = CtqmcGpu.from_problem(prob, nchains=nch, seed=61)
    src.warmup(600)
    # a pair on the empty state: annihilated first, or on the flavour that does not hybridise
    bad = _pair(prob.beta, nb - 1, 1, [2, 1] if code == 5 else [1, 2])
    src_cfgs = [src.get_config(c) for c in range(nch)]
    src_cfgs[where] = dict(bad, n=2, outer_sst=_outer(src, 0))
    src.get_config = lambda c: src_cfgs[c]
    path = str(tmp_path / "configs.npz")
    src.save_configs(path)
    pair = []
    for one_by_one in (False, True):
        g = CtqmcGpu.from_problem(prob, nchains=nch, seed=62)
        g.warmup(500)
        with pytest.raises(CtqmcError) as e:
            if one_by_one:
                for c in range(nch):
                    g.set_config(c, *[src_cfgs[c][k] for k in ORDER])
            else:
                g.load_configs(path)
        assert e.value.code == code
        pair.append(g)
    a, b = pair
    assert np.array_equal(a.chain_status()["status"], b.chain_status()["status"])
    for c in range(nch):
        x, y = a.get_config(c), b.get_config(c)
        for k in ORDER + (() if c == where else ("trace_log", "trace_sign", "det_log", "det_sign", "cfgsign")):
            assert np.array_equal(x[k], y[k]), (c, k)
        if c == where:
            continue
        for f in range(2 * nb):
            assert np.array_equal(a.get_minv(c, f), b.get_minv(c, f)), (c, f)
        x, y = a.moves_log(c, 150), b.moves_log(c, 150)
        assert all(np.array_equal(x[k], y[k]) for k in x.dtype.names if k != "pad"), c
    for g in (a, b, src):
        g.close()


@pytest.mark.parametrize("where", [10, 57])
def test_states_beyond_one_launch_are_kept(where, tmp_path):
    """60 chains of 4 x 200 pairs: the states to keep are more than one launch
    holds; refused in the first launch and in the last."""
    prob, nch = P.kanamori_2orb(beta=50.0, TaudiffMax=-1.0), 60
    nb = prob.nbands

    def crowd(shift, pairs=200):
        t = (np.arange(2 * pairs) + 0.5) * (prob.beta / (2 * pairs))
        fl = [np.sort(t + shift + 1e-3 * f) for f in range(2 * nb)]
        o = np.argsort(np.concatenate(fl), kind="stable")
        cat = lambda v: np.concatenate([v(f) for f in range(2 * nb)])[o]   # noqa: E731
        return dict(n=o.size, taus=np.concatenate(fl)[o], orbs=cat(lambda f: np.full(2 * pairs, f % nb)),
                    spins=cat(lambda f: np.full(2 * pairs, f // nb)), cas=cat(lambda f: np.tile([1, 2], pairs)))

    print("beyond one launch", where, flush=True)
    g = CtqmcGpu.from_problem(prob, nchains=nch, seed=71)
    outer = _outer(g, 0)
    paths = []
    for i, shift in enumerate((0.0, 0.01)):
        cfgs = [dict(crowd(shift + 1e-5 * c), outer_sst=outer) for c in range(nch)]
        if i == 1:
            cfgs[where] = dict(_pair(prob.beta, 0, 0, [2, 1]), n=2, outer_sst=outer)
        src = CtqmcGpu.from_problem(prob, nchains=nch, seed=1, capacity=2)
        src.get_config = lambda c: cfgs[c]
        paths.append(str(tmp_path / ("%d.npz" % i)))
        src.save_configs(paths[-1])
        src.close()
    g.load_configs(paths[0])
    look = [0, where - 1, where + 1, 51, 52, 53, nch - 1]
    before = {c: (g.get_config(c), [g.get_minv(c, f) for f in range(2 * nb)]) for c in look}
    with pytest.raises(CtqmcError) as e:
        g.load_configs(paths[1])
    assert e.value.code == 5
    for c in look:
        x, (y, minv) = g.get_config(c), before[c]
        kept = c > where
        assert np.array_equal(x["taus"], y["taus"]) == kept, c
        if kept:
            assert all(np.array_equal(x[k], y[k]) for k in x), c
            assert all(np.array_equal(g.get_minv(c, f), minv[f]) for f in range(2 * nb)), c
    g.close()
