"""The projective QR, Q and inverse (csrc/factor.hip on tall matrices) on both sides of their lines: four and eight waves
(N up to 256 and 512), eight tiles a wave (N above 512), the inverse with four and eight waves (ne up to 256
and above), remainders in rows and columns.  Bars as in test_gpu_proj."""
import numpy as np
import pytest

from sunhubbardmy_amd import chain_seed
from sunhubbardmy_amd.proj import ProjModel, ProjWalkers
from test_gpu_proj import BASE, run_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("la", [256, 258, 514])
def test_tall(la):
    run_parity(dict(BASE, lattice="chain", lb=1, la=la, beta=0.2, nwrap=1, mid_len=1, rv=1.5, nustock=64,
                    kmode="checkerboard"), nsweeps=1)


@pytest.mark.parametrize("n", [768, 770, 896, 898, 1022, 1024])
def test_tall_to_the_largest(n):
    """The rows of every tile of the eight-tile form, up to N = 1024 and an inverse of 512: Q, the span of Q, the inverse and the
    weight after one slice on a random Slater determinant P, against numpy on the same X = B P.

    Householder's bound for Q^H Q - 1 and Q Q^H X - X is N eps = 2e-13 of ones, taken with the inverse's condition number
    below ten as 1e-11."""
    w = ProjWalkers(ProjModel(lattice="chain", lb=1, la=n, beta=0.1, dtau=0.1, rv=0.0, rhub=4.0, nflr=2, nwrap=1, mid_len=1,
                              nustock=64, kmode="dense", seed=chain_seed(n)))
    rng = np.random.default_rng(n)
    P = np.linalg.qr(rng.standard_normal((n, n // 2)) + 1j * rng.standard_normal((n, n // 2)))[0]
    w.init_conf()
    w.set_proj(0, P)
    w.sweep_start_0b()
    t = w.tables[0]
    urt = np.asarray(t["urt"]).reshape(n, n)
    X = urt @ (t["u"]["bmat"][w.get_uconf().reshape(-1) - 1][:, None] * (urt @ P))
    ul, ur, inv = w.state()
    assert np.array_equal(ul, P.conj().T)
    R = ur.conj().T @ X
    scale = np.abs(np.diag(R)).max()
    print("n", n, "unitary %.1e" % np.abs(ur.conj().T @ ur - np.eye(n // 2)).max(), flush=True)
    assert np.abs(ur.conj().T @ ur - np.eye(n // 2)).max() < 1e-11
    assert np.abs(ur @ R - X).max() < 1e-11 * scale and np.abs(np.tril(R, -1)).max() < 1e-11 * scale
    assert np.abs(inv @ (ul @ ur) - np.eye(n // 2)).max() < 1e-11
    s, ld = np.linalg.slogdet(P.conj().T @ X)
    lw = w.diag()["logweightf"]
    assert abs(lw.real - ld) < 1e-9 and abs(np.exp(1j * lw.imag) - s) < 1e-9
    w.close()
