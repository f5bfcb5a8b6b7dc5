"""The chip-wide factorizations (csrc/factor.hip) at the edges of their tiles: 16-column panels with
and without a remainder, one and several panels, four and eight waves (N <= 256, N <= 512), alone
and in an uneven batch, where every chain ends at its own panel.

Bounds: Householder Q is unitary and Q R reproduces the matrix to about N eps ~ 1e-13 (columns
compared to their own size: they are graded); the LU's pivots are LAPACK's, so L U and the solution
carry the backward error of partial pivoting, 1e-12 of the right-hand side for these matrices
(growth and condition number below 1e3)."""
import ctypes

import numpy as np
import pytest
import scipy.linalg

from sunhubbardmy_amd import FTWalkers, Model, _lib

pytestmark = pytest.mark.gpu

SEL = {"W1": 2, "W2": 3, "W3": 4, "W4": 5, "U": 8, "V": 9}


class Batch:
    def __init__(self, sizes):
        self.sizes = sizes
        self.w = FTWalkers([Model(lattice="chain", la=n, beta=0.3, kmode="dense", nwrap=3, seed=k + 1)
                            for k, n in enumerate(sizes)])
        self.L = _lib.testing_lib()

    def put(self, name, c, a, pt=0):
        a = np.asfortranarray(a, dtype=np.complex128)
        assert self.L.sh_dbg_put(self.w._ctx, c, SEL[name], pt, a.ctypes.data_as(_lib.dp)) == 0

    def get(self, name, c, pt=0):
        a = np.zeros((self.sizes[c], self.sizes[c]), np.complex128, order="F")
        assert self.L.sh_dbg_get(self.w._ctx, c, SEL[name], pt, a.ctypes.data_as(_lib.dp)) == 0
        return a

    def vec(self, sel, c, size, pt=0, put=None):
        v = np.zeros(size) if put is None else np.ascontiguousarray(put, np.float64)
        f = self.L.sh_dbg_get if put is None else self.L.sh_dbg_put
        assert f(self.w._ctx, c, sel, pt, v.ctypes.data_as(_lib.dp)) == 0
        return v

    def op(self, code, *args):
        a = np.zeros(8, np.int32)
        a[:len(args)] = args
        assert self.L.sh_dbg_op(self.w._ctx, code, a.ctypes.data_as(_lib.ip)) == 0


CASES = [[n] for n in (2, 14, 16, 18, 32, 34, 62, 64, 66, 130, 144, 256, 258, 288, 400, 512)]
CASES += [[64, 16, 130, 2, 50], [30, 300, 64, 258]]


def rnd(n, rng):
    return rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))


@pytest.mark.parametrize("sizes", CASES)
def test_qr_and_q(sizes):
    b = Batch(sizes)
    rng = np.random.default_rng(len(sizes) + sizes[0])
    ref = []
    for c, n in enumerate(sizes):
        A, D = rnd(n, rng), np.exp(rng.uniform(-10, 10, n)) * rng.choice([-1.0, 1.0], n)
        b.put("W1", c, A)
        b.vec(100, c, n, 0, D)
        b.put("V", c, np.eye(n), 0)
        ref.append(A @ np.diag(D))
    b.op(4, 1, 0)
    for c, n in enumerate(sizes):
        U, V, D = b.get("U", c, 1), b.get("V", c, 1), b.vec(100, c, n, 1)
        print("n", n, "unitary %.1e" % np.abs(U.conj().T @ U - np.eye(n)).max(), flush=True)
        assert np.abs(U.conj().T @ U - np.eye(n)).max() < 1e-13
        err = np.abs(U @ np.diag(D) @ V - ref[c]).max(axis=0) / np.abs(ref[c]).max(axis=0)
        assert err.max() < 1e-12
        s, ld = np.linalg.slogdet(U)
        got = b.vec(103, c, 2, 1)
        assert abs(got[0] - ld) < 1e-10 and abs(np.exp(1j * got[1]) - s) < 1e-10
    b.w.close()


# Columns whose squared norm is still a number but |alpha - beta|^2 of their reflector, up to four times that, is beyond
# either end of the exponent range: its reciprocal is not representable below 2^-1024, its square not above
# 2^1024.  Squares near 2^-1074 are rounded to that absolute step: relative to nu^2 / n, the least a reflector meets,
# n 2^-1075 / nu^2 < 1e-13 at nu = 3e-155 and n = 34, so 1e-11 for the sums of them.
@pytest.mark.parametrize("n", [2, 18, 34])
@pytest.mark.parametrize("scale", [3e-155, 1.1e154])
def test_qr_at_the_ends_of_the_exponent_range(n, scale):
    b = Batch([n])
    rng = np.random.default_rng(n)
    A = np.eye(n) + 0.1 * rnd(n, rng) / np.sqrt(n)      # the diagonal carries most of a column's norm
    A /= np.linalg.norm(A, axis=0)
    b.put("W1", 0, A)
    b.vec(100, 0, n, 0, np.full(n, scale))
    b.put("V", 0, np.eye(n), 0)
    b.op(4, 1, 0)
    U, V, D = b.get("U", 0, 1), b.get("V", 0, 1), b.vec(100, 0, n, 1)
    assert np.abs(U.conj().T @ U - np.eye(n)).max() < 1e-11
    assert np.abs(U @ np.diag(D / scale) @ V - A).max() < 1e-11
    b.w.close()


@pytest.mark.parametrize("sizes", CASES)
def test_lu_and_solve(sizes):
    b = Batch(sizes)
    rng = np.random.default_rng(3 * len(sizes) + sizes[0])
    A = [rnd(n, rng) + 0.5 * np.sqrt(n) * np.eye(n) for n in sizes]
    X = [rnd(n, rng) for n in sizes]
    for c, n in enumerate(sizes):
        b.put("W3", c, A[c])
        b.put("W4", c, X[c])
    b.op(5)
    for c, n in enumerate(sizes):
        got, sc = b.get("W3", c), b.vec(104, c, 32)
        # zgetrf with pivots by |Re| + |Im|
        lu, piv = A[c].copy(), []
        for k in range(n):
            p = k + int(np.argmax(np.abs(lu[k:, k].real) + np.abs(lu[k:, k].imag)))
            piv.append(p)
            lu[[k, p]] = lu[[p, k]]
            lu[k + 1:, k] /= lu[k, k]
            lu[k + 1:, k + 1:] -= np.outer(lu[k + 1:, k], lu[k, k + 1:])
        scale = np.abs(lu).max()
        print("n", n, "LU %.1e" % (np.abs(got - lu).max() / scale), flush=True)
        assert np.abs(got - lu).max() / scale < 1e-11
        s, ld = np.linalg.slogdet(A[c])
        assert sc[14] == 0.0 and abs(sc[6] - ld) < 1e-9 and abs(np.exp(1j * sc[7]) - s) < 1e-9
        want = scipy.linalg.solve(A[c], X[c])
        assert np.abs(b.get("W4", c) - want).max() / np.abs(want).max() < 1e-10
    b.w.close()


@pytest.mark.parametrize("n,zero", [(18, 0), (34, 17), (130, 129), (288, 40)])
def test_lu_reports_the_first_zero_pivot(n, zero):
    b = Batch([n])
    A = np.eye(n, dtype=complex) + 0.1j * np.triu(np.ones((n, n)), 1)
    A[zero] = 0.0
    A[:, zero] = 0.0
    b.put("W3", 0, A)
    b.put("W4", 0, np.eye(n))
    b.op(5)
    assert b.vec(104, 0, 32)[14] == zero + 1
    b.w.close()
