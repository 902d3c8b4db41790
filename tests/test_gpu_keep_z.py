"""z through the caches or past them: the same bits.

A bunch of 1.05e7 particles alone keeps its z in the last cache, beside one of
2.1e7 both are streamed."""
import numpy as np
import pytest

from helpers import W

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,flags", [(8192, (True,) * 5), (4096, (True,) * 5), (65536, (True,) * 5),
                                      (16384, (True, False, True, True, False))])
def test_cached_z_equals_streamed(nb, flags):
    p = H.SimulationParameters.from_dict(W.ring_3gev_lattice(2, flags=flags))

    def bunch(n, seed):
        b = H.DeviceBunch(n)
        b.generate(seed, 4e-3, 3e6)
        return b

    def options():
        return H.TrackingOptions(seed=9, monitor=True, charge=2e-9, resonators=[W.RESONATOR_BB])
    alone, beside, big = bunch(10_500_001, 5), bunch(10_500_001, 5), bunch(21_000_000, 6)
    r = alone.evolve(p, nb, options())
    rs = H.batch_evolve([beside, big], [nb, 1024], [p, p], [options(), options()])
    for a, g in zip(alone.download(), beside.download()):
        assert np.array_equal(a, g)
    assert np.array_equal(r.monitor, rs[0].monitor) and r.E0 == rs[0].E0
    for b in (alone, beside, big):
        b.close()
