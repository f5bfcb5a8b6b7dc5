"""GPU parity: the HIP sweep (through the C ABI) against the CPU oracle on identical seeds.

Bar: identical accept/reject sequences (the HS field after every pass is
bit-identical), G within 1e-10 relative max-norm after every stabilization (nwrap), phase within
1e-10, observable bin sums within 1e-9 relative.
"""
import sys

import numpy as np
import pytest

import oracle
from sunhubbardmy_amd import FTWalkers, Model, chain_seed

pytestmark = pytest.mark.gpu

BASE = dict(lattice="square", la=4, lb=4, beta=2.0, dtau=0.1, rt=1.0, mu=0.0, rhub=4.0, nu=0.0, nflr=2,
            exact_hs=True, kmode="checkerboard", update="delay", nwrap=10, nublock=4)

CASES = {
    "square4_delay_checkerboard": {},
    "square4_fast_checkerboard": dict(update="fast"),
    "square4_delay_dense": dict(kmode="dense"),
    "square4_submatrix_checkerboard": dict(update="submatrix", nublock=5),
    "square6_su4_general_submatrix_dense": dict(la=6, lb=6, nflr=4, exact_hs=False, rhub=6.0, update="submatrix",
                                                 kmode="dense", nublock=8),
    "honeycomb3_delay_dense": dict(lattice="honeycomb", la=3, lb=3, kmode="dense", nublock=8),
    "honeycomb3_delay_checkerboard_nwrap7": dict(lattice="honeycomb", la=3, lb=3, nwrap=7, beta=1.6),
    "square4_su4_exact_delay": dict(nflr=4, exact_hs=True, rhub=6.0, nublock=3),
    "chain16_delay_checkerboard": dict(lattice="chain", la=16, lb=1, nublock=8),
    "chain10_fast_dense_mu": dict(lattice="chain", la=10, lb=1, kmode="dense", update="fast", mu=0.3),
    "cubic4_delay_checkerboard": dict(lattice="cubic", la=4, lb=4, lc=4, beta=1.0, nublock=8),
    "cubic4_submatrix_dense": dict(lattice="cubic", la=4, lb=4, lc=4, beta=0.8, kmode="dense", update="submatrix",
                                   nublock=8),
    # N = 400: seven blocks of sites, the last one of 16
    "square20_submatrix64_dense": dict(la=20, lb=20, beta=0.2, kmode="dense", update="submatrix", nublock=64,
                                       nwrap=2),
    # twenty slices between two stabilizations; the oracle pivots the first point's columns, the batch sorts them
    "square6_nwrap20": dict(la=6, lb=6, beta=4.0, nwrap=20, nublock=8),
    # above N = 512 every factorization is the one of a workgroup per chain
    "chain514_nwrap1": dict(lattice="chain", la=514, lb=1, beta=0.2, nwrap=1, nublock=8),
}


def relmax(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def run_parity(kw, nsweeps=2, chain=0):
    seed = chain_seed(chain)
    m = Model(seed=seed, **kw)
    say("case", kw, "seed", seed)
    w = FTWalkers([m])
    o = oracle.OracleChain(seed=seed, **kw)
    w.init_conf()
    o.init_conf()
    assert np.array_equal(w.get_conf(), o.conf), "initial HS field differs"
    w.sweep_start_0b()
    o.sweep_start()
    assert relmax(w.G(), o.G) < 1e-10
    cap = 4 * o.nst * nsweeps + 4
    w.set_trace(cap)
    o.set_trace(cap)
    for s in range(nsweeps):
        for p in ("b0", "0b"):
            getattr(w, "sweep_" + p)(True, True)
            getattr(o, "sweep_" + p)(True, True)
            say("  sweep", s, p)
            cw, co = w.get_conf(), o.conf
            assert np.array_equal(cw, co), "HS field differs after pass %d %s (%d sites)" % (s, p, (cw != co).sum())
    tw, to = w.trace(), o.trace()
    assert len(tw) == len(to) and len(tw) > 0
    for k in range(len(tw)):
        assert relmax(tw[k], to[k]) < 1e-10, "G differs at stabilization %d: %g" % (k, relmax(tw[k], to[k]))
    dw, do = w.diag(), o.diag()
    assert abs(dw["phase"] - do["phase"]) < 1e-10
    assert dw["accepted"] == do["accepted"] and dw["tried"] == do["tried"]
    assert dw["max_wrap_error"] < 1e-8
    ow, oo = w.obs(), o.obs()
    assert ow["nobs"] == oo["nobs"]
    for k in ("sign", "density", "ekin", "dblocc", "s_stag"):
        assert abs(ow[k] - oo[k]) <= 1e-9 * max(1.0, abs(oo[k])), k
    w.close()
    return dw, do


@pytest.mark.parametrize("name", list(CASES))
def test_sweep_parity(name):
    kw = dict(BASE)
    kw.update(CASES[name])
    run_parity(kw, nsweeps=1 if name == "chain514_nwrap1" else 2)


@pytest.mark.parametrize("name", ["square4_delay_checkerboard", "square6_su4_general_submatrix_dense"])
def test_the_update_and_its_depth_change_nothing(name):
    """One form of the update serves every build: a sweep has the same bits whatever update and nublock are."""
    kw = dict(BASE)
    kw.update(CASES[name])
    got = []
    for update, nublock in (("delay", 1), ("delay", 32), ("submatrix", 2), ("submatrix", 64), ("fast", 1)):
        w = FTWalkers([Model(seed=chain_seed(0), **dict(kw, update=update, nublock=nublock))])
        w.init_conf()
        w.sweep_start_0b()
        w.sweep(True, True)
        got.append((w.get_conf(), w.G(), w.diag(), w.obs()))
        w.close()
    for conf, G, diag, obs in got[1:]:
        assert np.array_equal(conf, got[0][0]) and np.array_equal(G, got[0][1])
        assert diag == got[0][2] and obs == got[0][3]


@pytest.mark.parametrize("la,lb,beta", [(4, 4, 8.0), (6, 6, 4.0), (8, 8, 8.0)])
def test_first_point_of_many_slices(la, lb, beta):
    """The first point of a chain, sorted by column norms here and column-pivoted in the oracle, with 10 to 80
    slices in it: G at the start of a sweep against the oracle's with a stabilization at every slice, no
    further off than four times what the pivoted form is (1e-14 at 10 slices, 1e-9 to 1e-8 at 80)."""
    kw = dict(BASE, la=la, lb=lb, beta=beta, nublock=8)
    ref = oracle.OracleChain(seed=chain_seed(3), **dict(kw, nwrap=1))
    ref.init_conf()
    ref.sweep_start()
    for nwrap in (10, 20, 40, 80):
        if nwrap > round(beta / 0.1):
            continue
        kw["nwrap"] = nwrap
        w, o = FTWalkers([Model(seed=chain_seed(3), **kw)]), oracle.OracleChain(seed=chain_seed(3), **kw)
        w.init_conf()
        o.init_conf()
        w.sweep_start_0b()
        o.sweep_start()
        ew, eo = relmax(w.G(), ref.G), relmax(o.G, ref.G)
        say("  nwrap", nwrap, "error %.1e, pivoted %.1e" % (ew, eo))
        assert ew < 4 * eo + 1e-13
        w.close()


def test_sweep_parity_metric_shape_short():
    # the bench shape (16x16) at a short beta: four blocks of sites, factorizations of sixteen panels
    kw = dict(BASE)
    kw.update(la=16, lb=16, beta=1.0, rhub=6.0, nublock=32, nwrap=5)
    run_parity(kw, nsweeps=1)


def test_uneven_batch_matches_single_chains():
    """Chains of different N and lattices in one batch (one launch per kernel for all of them):
    every chain's field and G equal its own oracle run with the same seed."""
    base = dict(beta=1.0, dtau=0.1, rhub=4.0, nflr=2, kmode="checkerboard", update="delay", nwrap=5, nublock=4)
    shapes = [dict(lattice="square", la=4, lb=4), dict(lattice="honeycomb", la=3, lb=3),
              dict(lattice="square", la=6, lb=6), dict(lattice="chain", la=10, lb=1)]
    models = [Model(seed=chain_seed(c), **base, **sh) for c, sh in enumerate(shapes)]
    say("uneven batch", [m.lattice for m in models])
    w = FTWalkers(models)
    oracles = [oracle.OracleChain(seed=chain_seed(c), **base, **sh) for c, sh in enumerate(shapes)]
    w.init_conf()
    for o in oracles:
        o.init_conf()
    w.sweep_start_0b()
    for o in oracles:
        o.sweep_start()
    for p in ("b0", "0b"):
        getattr(w, "sweep_" + p)(True, True)
        for o in oracles:
            getattr(o, "sweep_" + p)(True, True)
    for c, o in enumerate(oracles):
        assert np.array_equal(w.get_conf(c), o.conf), c
        assert relmax(w.G(c), o.G) < 1e-10, c
        ow, oo = w.obs(c), o.obs()
        for k in ("density", "ekin", "dblocc", "s_stag"):
            assert abs(ow[k] - oo[k]) <= 1e-9 * max(1.0, abs(oo[k])), (c, k)
    w.close()
