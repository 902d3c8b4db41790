"""The convolution at every block size the LDS holds, beside the oracle's FFT."""
import numpy as np
import pytest

from helpers import COORD_RTOL, W, normwise
from oracle import oracle as O

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fft_block", [64, 128, 512, 1024, 2048, 4096])
@pytest.mark.parametrize("nb", [9000, 4097])
def test_block_sizes(nb, fft_block):
    n = 20_001
    z0, e0 = O.generate_gaussian(5, 0.0, 4e-3, 0.0, 3e6, n)
    p = W.ring_3gev_lattice(2)
    zr, er, rr = O.evolve(z0, e0, nb, p, seed=3, charge=2e-9, resonators=[W.RESONATOR_BB])
    b = H.DeviceBunch(n)
    b.upload(z0, e0)
    r = b.evolve(H.SimulationParameters.from_dict(p), nb,
                 H.TrackingOptions(seed=3, charge=2e-9, resonators=[W.RESONATOR_BB], fft_block=fft_block))
    z, e = b.download()
    b.close()
    assert normwise(z, zr) <= COORD_RTOL and normwise(e, er) <= COORD_RTOL
    assert r.E0 == pytest.approx(rr.E0, rel=1e-14)
