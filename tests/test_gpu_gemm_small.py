"""The 32 x 32 form of the chains' products (csrc/gemm_small.h) at the edges of its tiles and of its steps of
64 along K, one chain and uneven batches, and on both sides of the launch rule; batches of more than 32 chains that are no multiple
of eight, whose last group has places without a chain (45 of N = 30 in 32 x 32 tiles, 250 of N = 62 in 64 x 64 tiles).

Bound: sums of N products of entries of order one, 4 N eps of N's worst sum ~ 1e-13 of the largest entry."""
import ctypes

import numpy as np
import pytest

from sunhubbardmy_amd import FTWalkers, Model, _lib

pytestmark = pytest.mark.gpu

SEL = {"W1": 2, "W2": 3, "W3": 4}


@pytest.mark.parametrize("sizes", [[2], [14], [30], [32], [34], [62], [64], [66], [96], [98], [130], [288], [2, 66, 34, 130],
                                   [254] * 15, [256] * 16, [30] * 45, [2, 66, 34, 130, 32] * 7,
                                   [62] * 250])
def test_gemm_edges(sizes):
    w = FTWalkers([Model(lattice="chain", la=n, beta=0.3, kmode="dense", nwrap=3, seed=k + 1) for k, n in enumerate(sizes)])
    L = _lib.testing_lib()
    rng = np.random.default_rng(sum(sizes))
    A, B = ([np.asfortranarray(rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) for n in sizes] for _ in "ab")
    for c in range(len(sizes)):
        assert L.sh_dbg_put(w._ctx, c, SEL["W1"], 0, A[c].ctypes.data_as(_lib.dp)) == 0
        assert L.sh_dbg_put(w._ctx, c, SEL["W2"], 0, B[c].ctypes.data_as(_lib.dp)) == 0
    for code, f in ((0, lambda a, b: a @ b), (1, lambda a, b: a.conj().T @ b), (2, lambda a, b: a @ b.conj().T)):
        a8 = np.zeros(8, np.int32)
        assert L.sh_dbg_op(w._ctx, code, a8.ctypes.data_as(_lib.ip)) == 0
        for c, n in enumerate(sizes):
            C = np.zeros((n, n), np.complex128, order="F")
            assert L.sh_dbg_get(w._ctx, c, SEL["W3"], 0, C.ctypes.data_as(_lib.dp)) == 0
            ref = f(A[c], B[c])
            assert np.abs(C - ref).max() < 1e-13 * np.abs(ref).max(), (code, c, n)
    w.close()
