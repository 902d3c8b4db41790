"""Particles of windowed histograms through the caches or past them: the same bits.

Alone, the bunch fits the last cache; beside another of its kind, both are
streamed.  The second batch ends with the bunch alone again, which then goes back
through the caches."""
import numpy as np
import pytest

from helpers import W

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("other_turns", [3, 1])
@pytest.mark.parametrize("nb,flags", [(65536, (True,) * 5), (131073, (True,) * 5),
                                      (65536, (True, False, False, True, True))])
def test_cached_equals_streamed(nb, flags, other_turns):
    def params(turns):
        return H.SimulationParameters.from_dict(W.ring_3gev_lattice(turns, flags=flags))

    def bunch(n, seed):
        b = H.DeviceBunch(n)
        b.generate(seed, 4e-3, 3e6)
        return b

    def options():
        return H.TrackingOptions(seed=9, monitor=True, charge=2e-9, resonators=[W.RESONATOR_BB])
    alone, beside, other = bunch(6_000_001, 5), bunch(6_000_001, 5), bunch(9_000_000, 6)
    r = alone.evolve(params(3), nb, options())
    rs = H.batch_evolve([beside, other], [nb, 65536], [params(3), params(other_turns)], [options(), options()])
    for a, g in zip(alone.download(), beside.download()):
        assert np.array_equal(a, g)
    assert np.array_equal(r.monitor, rs[0].monitor) and r.E0 == rs[0].E0
    for b in (alone, beside, other):
        b.close()
