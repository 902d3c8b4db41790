"""The E0 update by one workgroup per bunch against the one by slices, bit for bit.

Alone, a bunch of few slices takes the first; beside one of ten slices without a
deposit, both take the second: one to eight slices of interpolation sums, and
deposits of several rounds of cells."""
import numpy as np
import pytest

from helpers import W

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nb", [(3, 9000), (2_047, 9000), (131_072, 9000), (131_075, 9000), (400_001, 9000),
                                  (1_048_576, 9000), (20_000, 2), (20_000, 1025), (20_000, 4096), (20_000, 4098),
                                  (20_000, 5121), (300_001, 5700)])
def test_whole_equals_slices(n, nb):
    p = H.SimulationParameters.from_dict(W.ring_3gev_lattice(3))

    def bunch(n, seed):
        b = H.DeviceBunch(n)
        b.generate(seed, 4e-3, 3e6)
        return b

    def options():
        return H.TrackingOptions(seed=9, tile_pairs=1, monitor=True, charge=2e-9, bin_whole=-1,
                                 resonators=[W.RESONATOR_BB])
    alone, beside, big = bunch(n, 5), bunch(n, 5), bunch(1_250_000, 6)
    r = alone.evolve(p, nb, options())
    rs = H.batch_evolve([beside, big], [nb, 9000], [p, p], [options(), options()])
    for a, g in zip(alone.download(), beside.download()):
        assert np.array_equal(a, g)
    assert np.array_equal(r.monitor, rs[0].monitor, equal_nan=True) and r.E0 == rs[0].E0
    for b in (alone, beside, big):
        b.close()
