"""The stocks of the projective submatrix-LR update (csrc/stock_kernels.hip) at the edges of their tiles: stocks of
one to four register tiles of 16 sites, with and without a remainder, one and several 32-wide tiles of
the occupied space, for the bond field (a chain of 2 m sites has two families of m bonds) and the on-site field.
Bars as in test_gpu_proj: fields and acceptance counts identical to the oracle's, G within 1e-10."""
import pytest

from test_gpu_proj import BASE, run_parity

pytestmark = pytest.mark.gpu

KW = dict(BASE, lattice="chain", lb=1, beta=0.4, nwrap=2, mid_len=1, kmode="checkerboard")


@pytest.mark.parametrize("la,nustock", [(16, 14), (30, 16), (34, 32), (62, 18), (66, 34), (96, 48), (140, 64)])
def test_bond_stocks(la, nustock):
    run_parity(dict(KW, la=la, nustock=nustock, rv=2.0), nsweeps=1)


@pytest.mark.parametrize("la,nustock", [(16, 16), (34, 18), (62, 30), (66, 64), (98, 48), (130, 50)])
@pytest.mark.parametrize("nflr", [2, 4])
def test_site_stocks(la, nustock, nflr):
    run_parity(dict(KW, la=la, nustock=nustock, rv=0.0, rhub=4.0, nflr=nflr), nsweeps=1)


def test_site_stock_ratios_beyond_the_exponent_range():
    """The first stock of 24 flavours at U = -8 from a random field: its accepted ratios multiply to more than 1e154."""
    run_parity(dict(KW, la=66, nustock=64, rv=0.0, rhub=-8.0, nflr=24, exact_hs=False), nsweeps=1)
