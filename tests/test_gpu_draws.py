"""The generator's stream (csrc/kernels.hip, sfmt_refill) around the ends of its 624-number blocks: the initial field of
4 * ltrot numbers, then a sweep's draws, against the oracle's, number by number through the fields."""
import numpy as np
import pytest

import oracle
from sunhubbardmy_amd import FTWalkers, Model, chain_seed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ltrot", [2, 155, 156, 157, 312, 470])
def test_draws(ltrot):
    kw = dict(lattice="square", la=2, lb=2, beta=0.01 * ltrot, dtau=0.01, rhub=4.0, nwrap=10, kmode="checkerboard")
    w = FTWalkers([Model(seed=chain_seed(c + 2), **kw) for c in range(2)])
    os_ = [oracle.OracleChain(seed=chain_seed(c + 2), **kw) for c in range(2)]
    w.init_conf()
    print("ltrot", ltrot, flush=True)
    for c, o in enumerate(os_):
        o.init_conf()
        assert np.array_equal(w.get_conf(c), o.conf)
        o.sweep_start()
        o.sweep_b0(True, False)
    w.sweep_start_0b()
    w.sweep_b0(True, False)
    for c, o in enumerate(os_):
        assert np.array_equal(w.get_conf(c), o.conf)
    w.close()
