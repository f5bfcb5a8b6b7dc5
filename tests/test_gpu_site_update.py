"""The on-site update of one slice (csrc/update_kernels.hip) against sequential rank-1 updates in
numpy: the sizes around the edges of its blocks (16-site register tiles, 64-site blocks, 64-wide
panels and tiles), one chain alone and chains of uneven size in a batch, two and four field
components, one to four flavours.

The field must be the same site by site.  G after the slice: every accepted site multiplies the
rounding by at most about |delta / ratio| < 1e2 of entries of order one, and the product form
differs from the sequential one in the order of N sums, so 1e-10 of the largest entry (the
project's bar for G) leaves two orders."""
import ctypes

import numpy as np
import pytest

import oracle
from sunhubbardmy_amd import FTWalkers, Model, _lib, chain_seed

pytestmark = pytest.mark.gpu

SIZES = [2, 14, 16, 18, 32, 34, 48, 50, 62, 64, 66, 80, 96, 126, 128, 130, 192, 200, 260]


def update(hs, nflr, G, conf, u):
    """dqmc_update.f90 of one slice; (G, field, accepted, phase), and the smallest distance of a
    decision from its threshold."""
    G, conf, phase, acc, margin = G.copy(), conf.copy(), 1.0 + 0j, 0, 1.0
    lc = hs["lcomp"]
    for s in range(G.shape[0]):
        is_ = conf[s] - 1
        fl = int(np.ceil(u[s, 0] * (lc - 1)))
        isp = (is_ + fl) % lc
        db = hs["delta_bmat"][fl - 1, is_]
        r1 = 1.0 + (1.0 - G[s, s]) * db
        rt = r1 ** nflr * hs["gaml"][isp] / hs["gaml"][is_] * hs["phase_ratio"][fl - 1, is_]
        re = abs((rt * phase).real / phase.real)
        margin = min(margin, abs(re - u[s, 1]))
        if re > u[s, 1]:
            acc += 1
            phase *= rt / abs(rt)
            row = G[s].copy()
            row[s] -= 1.0
            G += np.outer(G[:, s] * (db / r1), row)
            conf[s] = isp + 1
    return G, conf, acc, phase, margin


def check(sizes, **kw):
    models = [Model(lattice="chain", la=n, beta=0.3, dtau=0.1, kmode="dense", nwrap=3, seed=chain_seed(7 * k + n), **kw)
              for k, n in enumerate(sizes)]
    w = FTWalkers(models)
    L = _lib.testing_lib()

    def op(code, *args):
        a = np.zeros(8, np.int32)
        a[:len(args)] = args
        assert L.sh_dbg_op(w._ctx, code, a.ctypes.data_as(_lib.ip)) == 0
    rng = np.random.default_rng(sum(sizes))
    want = []
    op(11)
    for c, n in enumerate(sizes):
        hs = w.tables[c]["hs"]
        G = np.asfortranarray(0.5 * np.eye(n) + 0.4 * (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) /
                              np.sqrt(2 * n))
        conf = rng.integers(1, hs["lcomp"] + 1, size=(3, n)).astype(np.int32)
        w.set_conf(conf, c)
        assert L.sh_dbg_put(w._ctx, c, 0, 0, G.ctypes.data_as(_lib.dp)) == 0
        u = oracle.sfmt_stream(models[c].seed, 6 * n).reshape(3, n, 2)
        want.append((update(hs, models[c].nflr, G, conf[1], u[2]), conf))
    op(10, 2, 2)                        # slice 2 with the uniforms of the pass's third slice
    for c, n in enumerate(sizes):
        (G, field, acc, phase, margin), conf = want[c]
        got, d = w.get_conf(c), w.diag(c)
        print("n", n, kw, "accepted", acc, "margin %.1e" % margin, flush=True)
        assert margin > 1e-9            # no tie: the decisions are determined
        assert np.array_equal(got[1], field) and np.array_equal(got[[0, 2]], conf[[0, 2]])
        assert d["accepted"] == acc and d["tried"] == n
        assert abs(d["phase"] - phase) < 1e-10
        assert np.abs(w.G(c) - G).max() < 1e-10 * np.abs(G).max()
    w.close()


@pytest.mark.parametrize("n", SIZES)
def test_one_chain(n):
    check([n], rhub=4.0, update="delay", nublock=8)


@pytest.mark.parametrize("kw", [dict(rhub=4.0, update="fast"), dict(rhub=-3.0, update="delay", nublock=16),
                                dict(rhub=6.0, nflr=4, exact_hs=False, update="submatrix", nublock=32),
                                dict(rhub=2.0, nflr=1, exact_hs=False, update="submatrix", nublock=64)])
def test_uneven_batch(kw):
    check([64, 14, 130, 48, 66, 200, 2], **kw)
    check([62, 16, 30], **kw)


# A field far from the weights' maximum: the accepted ratios of a block multiply to 1e200 (12 flavours, U = -8; two
# flavours, U = -120) and 1e312 (U = -16; -240), where the decisions and the phase need only their direction.
@pytest.mark.parametrize("sizes", [[64], [130], [64, 130, 34]])
@pytest.mark.parametrize("nflr,u", [(12, -8.0), (12, -16.0), (2, -120.0), (2, -240.0)])
def test_ratios_beyond_the_exponent_range(nflr, u, sizes):
    check(sizes, rhub=u, nflr=nflr, exact_hs=False, update="delay", nublock=16)
