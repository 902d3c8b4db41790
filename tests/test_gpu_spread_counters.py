"""Histogram and deposit counters with gaps between their lines.

From 32 tiles on a bunch's global counters use every other 128 bytes.  The same
bunch in 33 and in 17 tiles gets the same counts, and the same coordinates to the
rounding of its sums over tiles, at numbers of bins around a line's counters."""
import numpy as np
import pytest

from helpers import COORD_RTOL, W, normwise

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("update_E0", [True, False])   # with and without the deposit
@pytest.mark.parametrize("nb", [1, 2, 15, 16, 17, 31, 32, 33, 100, 1025, 2049, 4097, 9000])
def test_spread_counters(nb, update_E0):
    n = 67_001
    p = H.SimulationParameters.from_dict(W.ring_3gev_lattice(4, flags=(True, True, update_E0, True, True)))
    out = []
    for tile_pairs in (1, 2):
        b = H.DeviceBunch(n)
        b.generate(5, 4e-3, 3e6)
        r = b.evolve(p, nb, H.TrackingOptions(seed=9, tile_pairs=tile_pairs, monitor=True, charge=2e-9,
                                              resonators=[W.RESONATOR_BB], bin_half_width_sigmas=2.5))
        out.append((*b.download(), r))
        b.close()
    (z1, e1, r1), (z2, e2, r2) = out
    assert normwise(z1, z2) <= COORD_RTOL and normwise(e1, e2) <= COORD_RTOL
    assert r1.E0 == pytest.approx(r2.E0, rel=1e-14)
    assert np.max(np.abs(r1.monitor[:, 3] - r2.monitor[:, 3])) <= 1   # the grid's ends differ in the last place
