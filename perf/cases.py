"""The work this framework does, as cases that can be timed and compared.

Every case is one pass through the public entry points: a Monte Carlo sweep of a batch of
finite-temperature chains (``FTWalkers``), of projective chains (``ProjWalkers``), the
time-displaced measurement of a fixed field, or an epoch of the effective action's training.
A sweep returns the bins of the pass and the chains' whole state (the HS fields, and G unless a
batch's G's together are more than a program would fetch after every sweep).

``exact`` restates a pass in numpy (complex128) or torch (float64) where that takes seconds: the
Markov chain of one small SU(2) lattice, site by site with G rebuilt at every slice, the
equal-time G of a fixed field, and the network's training.
"""
import math

import numpy as np
import torch

from sunhubbardmy_amd import FTWalkers, Model, chain_seed
from sunhubbardmy_amd.learned import NWEIGHTS, EffectiveAction
from sunhubbardmy_amd.proj import ProjModel, ProjWalkers

G_BYTES = 64 << 20      # a batch whose G's are larger than this together keeps them on the device


# ---- the cases ---------------------------------------------------------------------------------
def ft(name=None, **kw):
    """A batch of finite-temperature chains.  ``sizes`` lists la x lb * chains, e.g. "8x8*32"."""
    c = dict(kind="ft", lattice="square", sizes="4x4*1", u=4.0, v=0.0, beta=4.0, flavours=2, exact_hs=True,
             kinetic="checkerboard", update="delay", depth=0, nprop=0, graphs=False)
    c.update(kw)
    return dict(name=name, **c) if name else c


def proj(name=None, **kw):
    """A batch of projective chains; ``beta`` is the projection length."""
    c = dict(kind="proj", lattice="honeycomb", sizes="6x6*1", u=0.0, v=1.2, beta=10.0, kinetic="dense",
             update="submatrix_lr")
    c.update(kw)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one chain of the smallest lattice in use, with the plain fast update: every launch and
        # every serial step counts (what one rank of a first trial run does)
        ft("ft 4x4, one chain, fast", sizes="4x4*1", beta=4.0, update="fast"),
        # sixteen chains of an ordinary small lattice, as on a 16-core node, replayed graphs, the
        # default delay depth
        ft("ft 8x8, 16 chains", sizes="8x8*16", beta=6.0, graphs=True),
        # the headline workload: 256 chains at 16x16, beta = 8, delay depth 32
        ft("ft 16x16, 256 chains, delay", sizes="16x16*256", u=6.0, beta=8.0, depth=32),
        # a single walker of a larger honeycomb lattice with the dense kinetic term: one chain
        # has the whole GPU
        ft("ft honeycomb 12, one chain", lattice="honeycomb", sizes="12x12*1", beta=10.0, depth=32, kinetic="dense"),
        # chains of three lattices in one batch, SU(4) with the four-component field, the FFT
        # kinetic term and the submatrix update
        ft("ft SU(4) uneven, 72 chains", sizes="8x8*32 12x12*24 16x16*16", u=6.0, beta=8.0, flavours=4, exact_hs=False,
           kinetic="fft", update="submatrix", depth=32, graphs=True),
        # block proposals of 64 attempts on top of the local sweep, N = 400, few chains
        ft("ft 20x20, block proposals", sizes="20x20*16", u=6.0, beta=12.0, depth=64, nprop=64),
        # the t-U-V model: bond and on-site fields, ragged N = 72, dense kinetic term
        ft("ft t-U-V honeycomb 6", lattice="honeycomb", sizes="6x6*16", u=2.0, v=0.6, beta=3.0, kinetic="dense",
           flavours=2),
        # the projective t-V workload's lattice (N = 648, 324 particles), a shorter projection
        proj("proj t-V honeycomb 18, 8 chains", sizes="18x18*8", beta=3.0),
        # an ordinary projective run of a small lattice, a few chains
        proj("proj t-V honeycomb 6, 4 chains", sizes="6x6*4", beta=10.0),
        # the projective Hubbard model: on-site field, checkerboard kinetic term
        proj("proj Hubbard 10x10, 8 chains", lattice="square", sizes="10x10*8", u=4.0, v=0.0, beta=6.0,
             kinetic="checkerboard"),
        # restart from fields of a file, then the equal-time and time-displaced measurement of
        # them, no updates: the stabilization and the Green's functions
        dict(name="tau 12x12, 8 chains", kind="tau", lattice="square", sizes="12x12*8", u=4.0, v=0.0, beta=4.0,
             flavours=2, exact_hs=True, kinetic="checkerboard", update="delay", depth=0, nprop=0, graphs=False),
        # one epoch over the configurations of a training run (20480) in batches of 512
        dict(name="train, 20480 samples", kind="train", samples=20480, batch=512),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the kinds in the proportions in which they are listed, sizes over the range."""
    top = max(cost(c) for c in listed())
    while True:
        c = _draw(rng)
        if cost(c) <= top:
            return c


def _draw(rng):
    kind = rng.choice(["ft"] * 7 + ["proj"] * 3 + ["tau", "train"])
    if kind == "train":
        return dict(kind="train", samples=_spread(rng, 1000, 20480), batch=rng.choice([128, 256, 500, 512]))
    lattice = rng.choice(["square", "square", "honeycomb"]) if kind != "tau" else "square"

    def size():
        if lattice == "honeycomb":
            return "%dx%d" % (rng.randint(3, 12), rng.randint(3, 12))
        return "%dx%d" % (2 * rng.randint(2, 9), 2 * rng.randint(2, 9))
    if kind == "proj":
        tv = lattice == "honeycomb"
        return proj(lattice=lattice, sizes="%s*%d" % (size(), _spread(rng, 1, 16)), u=0.0 if tv else 4.0,
                    v=rng.choice([0.8, 1.2]) if tv else 0.0, beta=rng.choice([2.0, 3.0, 4.5]),
                    kinetic=rng.choice(["dense", "checkerboard"]))
    if kind == "tau":
        return ft(kind="tau", sizes="%s*%d" % (size(), _spread(rng, 1, 8)), beta=rng.choice([2.0, 3.0, 4.0]))
    parts = []
    for _ in range(rng.choice([1, 1, 1, 2])):
        parts.append("%s*%d" % (size(), _spread(rng, 1, 64)))
    su4 = rng.random() < 0.25
    kinetics = ["checkerboard", "checkerboard", "dense"] + (["fft"] if lattice == "square" else [])
    update, depth = rng.choice([("fast", 0), ("delay", 0), ("delay", 16), ("delay", 32), ("submatrix", 32),
                                ("submatrix", 16)])
    return ft(lattice=lattice, sizes=" ".join(parts), u=rng.choice([2.0, 4.0, 6.0]), beta=rng.choice([2.0, 3.0, 4.5, 6.0]),
              flavours=4 if su4 else 2, exact_hs=not su4, kinetic=rng.choice(kinetics), update=update, depth=depth,
              nprop=rng.choice([0, 0, 0, 16]) if not su4 else 0, graphs=rng.random() < 0.3)


def _sizes(case):
    """[(la, lb, chains)] of a case."""
    out = []
    for part in case["sizes"].split():
        ab, k = part.split("*")
        a, b = ab.split("x")
        out.append((int(a), int(b), int(k)))
    return out


def _sites(case, la, lb):
    return la * lb * (2 if case["lattice"] == "honeycomb" else 1)


def _nchains(case):
    return sum(k for _, _, k in _sizes(case))


def cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 10.0)


# ---- inputs ------------------------------------------------------------------------------------
def _seeds(case, seed):
    base = (int(seed) * 7919) % 100003
    return [chain_seed(1000 * base + c) for c in range(_nchains(case))]


def _ft_models(case, seed):
    seeds, out = _seeds(case, seed), []
    for la, lb, k in _sizes(case):
        for _ in range(k):
            out.append(Model(lattice=case["lattice"], la=la, lb=lb, beta=case["beta"], dtau=0.1, rhub=case["u"],
                             rv=case["v"], nflr=case["flavours"], exact_hs=case["exact_hs"], kmode=case["kinetic"],
                             update=case["update"], nublock=case["depth"], nwrap=10, seed=seeds[len(out)]))
    return out


def _fields(case, seed):
    """The fields of a saved run: independent +-1 values of every chain."""
    r = np.random.default_rng(int(seed))
    lt = int(round(case["beta"] / 0.1))
    return [r.integers(1, 3, size=(lt, _sites(case, la, lb))).astype(np.int32) for la, lb, k in _sizes(case)
            for _ in range(k)]


def _samples(case, seed):
    """Features and energies like those of a sweep: couplings near 0, an energy that depends on them."""
    r = np.random.default_rng(int(seed))
    f = 0.05 * r.standard_normal((case["samples"], 4))
    e = -0.9 + 0.4 * np.tanh(8.0 * f[:, 1]) - 0.3 * f[:, 2] + 0.01 * r.standard_normal(case["samples"])
    return np.concatenate([f, e[:, None]], axis=1)


def _weights(seed):
    r = np.random.default_rng(int(seed) + 17)
    w = np.zeros(NWEIGHTS, np.float32)
    o = 0
    for rows, cols in ((128, 4), (128, 0), (128, 128), (128, 0), (1, 128), (1, 0)):
        k = rows * max(cols, 1)
        if cols:
            w[o:o + k] = r.standard_normal(k) * math.sqrt(2.0 / (rows + cols))
        o += k
    return w


def prepare(case, seed):
    if case["kind"] == "train":
        net = EffectiveAction(capacity=case["samples"], seed=int(seed) % 100000 + 1)
        x = _samples(case, seed)
        net.set_weights(_weights(seed))
        net.set_norm(np.concatenate([x[:, :4].mean(0), x[:, :4].std(0), [x[:, 4].mean(), x[:, 4].std()]]))
        net.push_samples(x)
        return {"case": case, "net": net, "f": np.ascontiguousarray(x[:2048, :4])}
    if case["kind"] == "proj":
        seeds, models = _seeds(case, seed), []
        for la, lb, k in _sizes(case):
            for _ in range(k):
                models.append(ProjModel(lattice=case["lattice"], la=la, lb=lb, beta=case["beta"], dtau=0.1, rv=case["v"],
                                        rhub=case["u"], nflr=1 if case["v"] else 2, kmode=case["kinetic"], nwrap=10,
                                        rndness=1e-4, wrap_check=False, update=case["update"], seed=seeds[len(models)]))
        w = ProjWalkers(models)
        w.init_conf()
        w.set_trial()
        w.sweep_start_0b()
        return {"case": case, "w": w}
    w = FTWalkers(_ft_models(case, seed))
    if case["kind"] == "tau":
        for c, f in enumerate(_fields(case, seed)):
            w.set_conf(f, c)
        w.set_dyn()
        return {"case": case, "w": w}
    st = {"case": case, "w": w}
    w.set_graphs(case["graphs"])
    if case["nprop"]:
        w.set_neighbours()
    w.init_conf()
    w.sweep_start_0b()
    if case["nprop"]:
        # the effective action of a trained run is worth a few percent per coupling: a random
        # network on normalised features, energies of the batch's own scale
        net = EffectiveAction(capacity=16, seed=1)
        net.set_weights(_weights(seed))
        net.set_norm(np.array([0.0, 0.0, 0.0, 0.0, 0.05, 0.05, 0.05, 0.05, 0.0, 0.01]))
        w.set_proposal(net, nprop=case["nprop"], local_updates=True)
        st["net"] = net
    w.sweep(True, True)         # away from the random start, and every kind of pass seen once
    w.obs_all(reset=True)
    return st


# ---- one pass ----------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    if case["kind"] == "train":
        net = state["net"]
        loss = net.train(epochs=1, batch=case["batch"], lr=1e-3)
        return {"loss": loss, "weights": net.weights(), "energies": net.predict(state["f"])}
    w, nch = state["w"], state["w"].nchains
    if case["kind"] == "proj":
        w.sweep(True, True)
        obs = [w.obs(c) for c in range(nch)]
        w.reset_obs()
        out = {"obs": np.array([[o["sign"], o["density"], o["ekin"], o["dblocc"], o["s_stag"]] for o in obs])}
        get = w.get_conf if w.has_vconf else w.get_uconf
        out["field"] = np.stack([get(c) for c in range(nch)])
        out["G"] = np.stack([w.G(c) for c in range(nch)])
        return out
    if case["kind"] == "tau":
        w.sweep_start_0b()
        w.sweep_b0(False, True)
        obs, _ = w.obs_all(reset=True)
        w.reset_dyn_obs()
        w.push_stage()
        w.sweep_0b(False, False, True)
        w.pop_stage()
        return {"obs": obs, "G": [w.G(c) for c in range(nch)] if len(_sizes(case)) > 1 else
                np.stack([w.G(c) for c in range(nch)]), "znn": np.stack([w.dyn_obs(c)[0] for c in range(nch)])}
    w.sweep(True, True)
    obs, _ = w.obs_all(reset=True)
    out = {"obs": obs, "field": np.concatenate([w.get_conf(c).reshape(-1) for c in range(nch)])}
    if w.has_vconf:
        out["bonds"] = np.concatenate([w.get_confv(c).reshape(-1) for c in range(nch)])
    if sum(16 * t["ndim"] ** 2 for t in w.tables) <= G_BYTES:
        out["G"] = np.concatenate([w.G(c).reshape(-1) for c in range(nch)])
    return out


# ---- what a pass cannot do without -------------------------------------------------------------
def work(case):
    """Bytes: G read and written once per slice and pass, B products and chain points once per
    stabilization.  Flops: the rank-1 updates of the accepted flips (8 a N^3 per slice), dense
    kinetic products (32 N^3, 16 N^3 on the projective sweep's half-width matrices), 64 N^3 per stabilization."""
    if case["kind"] == "train":
        return {"bytes": 40.0 * case["samples"] + 12.0 * NWEIGHTS, "flops": 6.0 * NWEIGHTS * case["samples"]}
    nbytes = flops = 0.0
    lt = round(case["beta"] / 0.1)
    for la, lb, k in _sizes(case):
        n = float(_sites(case, la, lb))
        if case["kind"] == "proj":
            # N x N/2 propagators; every field value is a row (bond: two rows) of a rank update of
            # the (N/2)^2 inverse, plus its row of the propagated product
            fields = n if case["u"] else 1.5 * n
            rows = 1.0 if case["u"] else 2.0
            kin = 16.0 * n ** 3 if case["kinetic"] == "dense" else 0.0
            flops += k * 2 * lt * (kin + 8.0 * fields * rows * (n * n / 4 + 0.5 * n * n / 4) + 8.0 * n ** 3 / 10)
            nbytes += k * 2 * lt * 2 * 16.0 * n * n
            continue
        passes = 2.0 if case["kind"] == "ft" else 4.0
        acc = 0.0 if case["kind"] == "tau" else 0.65 if case["flavours"] == 2 else 0.35
        kin = 32.0 * n ** 3 if case["kinetic"] == "dense" else 0.0
        flops += k * passes * lt * (8.0 * acc * n ** 3 + kin + 6.4 * n ** 3)
        nbytes += k * passes * lt * 32.0 * n * n
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """The Metropolis decisions are the same in every correct implementation (a tie within rounding
    is a 1e-10 event per pass); G and the bins differ by the rounding that the stabilization and
    the propagation over nwrap slices amplify: up to 7e-12 against the 64-bit restatement, 3e-12
    between two depths of the updates."""
    if case["kind"] == "train":
        # float32: 3e-7 in the loss and 2e-7 in the weights against Adam in float64
        return {"rel": 1e-5, "max": 1e-3}
    if case["kind"] == "proj":
        # the projected overlap is the worse conditioned one: imaginary parts that vanish exactly
        # come out at 1e-10 of the result
        return {"rel": 1e-8, "max": 1e-6, "differ": 0.0}
    return {"rel": 1e-9, "max": 1e-7, "differ": 0.0}


# ---- the same in 64 bits, without the library --------------------------------------------------
def exact(case, seed):
    if case["kind"] == "train":
        return _exact_train(case, seed)
    sizes = _sizes(case)
    if case["kind"] == "tau" and sum(k * _sites(case, a, b) ** 3 * case["beta"] for a, b, k in sizes) < 2e8:
        g = [_g_zero(_slices(case, a, b, f)) for (a, b), f in
             zip([(a, b) for a, b, k in sizes for _ in range(k)], _fields(case, seed))]
        return {"obs": None, "G": g if len(sizes) > 1 else np.stack(g), "znn": None}
    if (case["kind"] == "ft" and len(sizes) == 1 and sizes[0][2] == 1 and case["lattice"] == "square" and
            case["kinetic"] != "fft" and case["flavours"] == 2 and case["exact_hs"] and not case["v"] and
            not case["nprop"] and _sites(case, *sizes[0][:2]) ** 2 * case["beta"] ** 2 <= 20000):
        return _exact_chain(case, seed)
    return None             # a sweep of these takes minutes in numpy


def _site(x, y, la, lb):
    return (x % la) * lb + y % lb


def _half_kinetic(case, la, lb):
    """(fwd, rev): exp(-dtau K / 2) of the square lattice as the families +x, +y, -x, -y applied
    first to last, and last to first; the dense exponential for both when kinetic is dense."""
    n = la * lb
    k = np.zeros((n, n))
    fams = []
    for dx, dy in ((1, 0), (0, 1), (-1, 0), (0, -1)):
        e = np.eye(n)
        for x in range(la):
            for y in range(lb):
                if (x + y) % 2 == 0:
                    a, b = _site(x, y, la, lb), _site(x + dx, y + dy, la, lb)
                    k[a, b] -= 1.0
                    k[b, a] -= 1.0
                    e[a, a] = e[b, b] = math.cosh(0.05)
                    e[a, b] = e[b, a] = math.sinh(0.05)
        fams.append(e)
    if case["kinetic"] == "dense":
        w, v = np.linalg.eigh(k)
        d = (v * np.exp(-0.05 * w)) @ v.T
        return d, d
    f1, f2, f3, f4 = fams
    return f4 @ f3 @ f2 @ f1, f1 @ f2 @ f3 @ f4


def _diag_v(case, field):
    alpha = math.acos(math.exp(-0.05 * case["u"]))
    return np.exp(1j * alpha * (2.0 * np.asarray(field) - 3.0))


def _slices(case, la, lb, field):
    fwd, rev = _half_kinetic(case, la, lb)
    return [(rev * _diag_v(case, f)[None, :]) @ fwd for f in field]


def _g_zero(mats):
    """(1 + mats[-1] ... mats[0])^-1 through a U D V product with a QR every 5 matrices."""
    n = mats[0].shape[0]
    u, d, v = np.eye(n, dtype=complex), np.ones(n), np.eye(n, dtype=complex)
    for s in range(0, len(mats), 5):
        for m in mats[s:s + 5]:
            u = m @ u
        u = u * d[None, :]
        p = np.argsort(-np.linalg.norm(u, axis=0))
        q, r = np.linalg.qr(u[:, p])
        d = np.abs(np.diag(r))
        v = (r / d[:, None]) @ v[p]
        u = q
    db, ds = np.maximum(d, 1.0), np.minimum(d, 1.0)
    uh = u.conj().T / db[:, None]
    return np.linalg.solve(uh + ds[:, None] * v, uh)


class _Sfmt:
    """SFMT19937 (Saito and Matsumoto) with the reference's linear seeding and (u + 1/2) / 2^32."""
    MASK = 0xbffffff6bffaffffddfecb7fdfffffef
    ALL = (1 << 128) - 1

    def __init__(self, seed):
        w = [seed & 0xffffffff]
        for i in range(1, 624):
            w.append((1812433253 * (w[-1] ^ (w[-1] >> 30)) + i) & 0xffffffff)
        par = (1, 0, 0, 0x13c9e684)
        if sum(bin(w[i] & par[i]).count("1") for i in range(4)) % 2 == 0:
            w[0] ^= 1       # the lowest set parity bit
        self.s = [w[4 * i] | w[4 * i + 1] << 32 | w[4 * i + 2] << 64 | w[4 * i + 3] << 96 for i in range(156)]
        self.out = []

    @staticmethod
    def _lanes(x, k, left):
        f = (lambda v: (v << k) & 0xffffffff) if left else (lambda v: v >> k)
        return sum(f(x >> (32 * i) & 0xffffffff) << (32 * i) for i in range(4))

    def _refill(self):
        s = self.s
        c, d = s[154], s[155]
        for i in range(156):
            a, b = s[i], s[(i + 122) % 156]
            r = a ^ (a << 8 & self.ALL) ^ (self._lanes(b, 11, False) & self.MASK) ^ (c >> 8) ^ self._lanes(d, 18, True)
            s[i], c, d = r, d, r
        self.out = [x >> (32 * l) & 0xffffffff for x in s for l in range(4)]

    def draw(self, count):
        got = []
        while len(got) < count:
            if not self.out:
                self._refill()
            take = min(count - len(got), len(self.out))
            got += self.out[:take]
            self.out = self.out[take:]
        return (np.array(got, np.float64) + 0.5) / 4294967296.0


def _exact_chain(case, seed):
    """The sweep of prepare() and the sweep of run() of one SU(2) chain: at every slice G is built
    anew from all slices and the sites are visited with rank-1 updates.  At half filling every
    ratio, phase included, is real and positive up to rounding."""
    la, lb, _ = _sizes(case)[0]
    n, lt = la * lb, int(round(case["beta"] / 0.1))
    rng = _Sfmt(_seeds(case, seed)[0])
    field = np.ceil(rng.draw(lt * n) * 2.0).astype(np.int64).reshape(lt, n)
    fwd, rev = _half_kinetic(case, la, lb)
    alpha = math.acos(math.exp(-0.05 * case["u"]))
    for half in range(4):
        u = rng.draw(2 * lt * n).reshape(lt, n, 2)
        for q in range(lt):
            s = lt - 1 - q if half % 2 == 0 else q
            dv = [_diag_v(case, f) for f in field]
            mats = [(rev * v[None, :]) @ fwd for v in dv]
            # cyclic product that ends with exp(V_s) exp(-dtau K / 2) of slice s
            g = _g_zero([rev] + mats[s + 1:] + mats[:s] + [dv[s][:, None] * fwd])
            for i in range(n):
                now = 2.0 * field[s, i] - 3.0
                delta = np.exp(-2j * alpha * now) - 1.0
                r1 = 1.0 + (1.0 - g[i, i]) * delta
                if abs((r1 * r1 * np.exp(2j * alpha * now)).real) > u[q, i, 1]:
                    row = g[i].copy()
                    row[i] -= 1.0
                    g = g + np.outer(g[:, i] * (delta / r1), row)
                    field[s, i] = 3 - field[s, i]
    return {"obs": None, "field": None, "G": _g_zero(_slices(case, la, lb, field)).reshape(-1)}


def _exact_train(case, seed):
    """One epoch of Adam in float64 over the library's shuffle (splitmix64, Fisher-Yates)."""
    x = _samples(case, seed)
    n, mask = len(x), (1 << 64) - 1
    s = (0x9E3779B97F4A7C15 * (int(seed) % 100000 + 1) + 0x632BE59BD9B4E019) & mask
    perm = list(range(n))

    def unif():
        nonlocal s
        s = (s + 0x9E3779B97F4A7C15) & mask
        z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        return float((z ^ (z >> 31)) >> 11) * 2.0 ** -53
    for k in range(n - 1, 0, -1):
        j = min(int(unif() * (k + 1)), k)
        perm[k], perm[j] = perm[j], perm[k]
    shapes = ((128, 4), (128,), (128, 128), (128,), (128,), (1,))
    w, o = torch.from_numpy(_weights(seed).astype(np.float64)), 0
    p = []
    for sh in shapes:
        k = int(np.prod(sh))
        p.append(w[o:o + k].reshape(sh).clone().requires_grad_(True))
        o += k
    t = torch.from_numpy(x)
    t = (t - torch.from_numpy(x.mean(0))) / torch.from_numpy(x.std(0))

    def net(f):
        return torch.tanh(torch.tanh(f @ p[0].T + p[1]) @ p[2].T + p[3]) @ p[4] + p[5]
    opt, total = torch.optim.Adam(p, lr=1e-3, betas=(0.9, 0.999), eps=1e-8), 0.0
    for b in range(0, n, case["batch"]):
        q = t[perm[b:b + case["batch"]]]
        opt.zero_grad()
        loss = ((net(q[:, :4]) - q[:, 4]) ** 2).mean()
        loss.backward()
        opt.step()
        total += float(loss.detach()) * len(q)
    with torch.no_grad():
        e = x[:, 4].mean() + x[:, 4].std() * net(t[:2048, :4])
        return {"loss": np.array([total / n]), "weights": torch.cat([v.detach().reshape(-1) for v in p]).numpy(),
                "energies": e.numpy()}
