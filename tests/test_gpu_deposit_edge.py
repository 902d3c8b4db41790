"""The largest grid whose bunches deposit in the turn pass, and the first whose E0
update takes the interpolation sums instead: 28 bytes of LDS per bin in 162816."""
import numpy as np
import pytest

from helpers import COORD_RTOL, W, normwise
from oracle import oracle as O

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [5087, 5088, 5813, 5814, 5815, 5816])
@pytest.mark.parametrize("n,tile_pairs", [(30_001, 0), (150_000, 3)])
def test_either_side_matches_the_oracle(nb, n, tile_pairs):
    turns = 4
    p = W.ring_3gev_lattice(turns)
    z0, e0 = O.generate_gaussian(21, 0.0, W.SIGMA_Z, 0.0, W.SIGMA_E, n)
    zr, er, rr = O.evolve(z0, e0, nb, p, seed=8, charge=2e-9, resonators=[W.RESONATOR_BB],
                          bin_half_width_sigmas=8.0)
    b = H.DeviceBunch(n)
    b.upload(z0, e0)
    r = b.evolve(H.SimulationParameters.from_dict(p), nb,
                 H.TrackingOptions(seed=8, charge=2e-9, resonators=[W.RESONATOR_BB], bin_half_width_sigmas=8.0,
                                   tile_pairs=tile_pairs))
    z, e = b.download()
    b.close()
    assert normwise(z, zr) <= COORD_RTOL and normwise(e, er) <= COORD_RTOL
    assert r.E0 == pytest.approx(rr.E0, rel=1e-14)
