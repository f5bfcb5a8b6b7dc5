"""The projective QR, Q and inverse (csrc/factor.hip on tall matrices) on both sides of their lines: four and eight waves
(N up to 256 and 512), eight tiles a wave (N above 512), the inverse with four and eight waves (ne up to 256
and above), remainders in rows and columns.  Bars as in test_gpu_proj."""
import pytest

from test_gpu_proj import BASE, run_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("la", [256, 258, 514])
def test_tall(la):
    run_parity(dict(BASE, lattice="chain", lb=1, la=la, beta=0.2, nwrap=1, mid_len=1, rv=1.5, nustock=64,
                    kmode="checkerboard"), nsweeps=1)
