"""The all-flags pass with a partial window of P, its gathers before or after the
prefetch: the bits of the pass for any flags (which a bunch without the
excitation in the batch asks for), at numbers of bins on both sides of the line
(31656 and 31657) and up to the last with 32-bit counts."""
import numpy as np
import pytest

from helpers import W

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [14001, 31655, 31656, 31657, 31658, 32768, 34560, 34561, 40699, 40700])
@pytest.mark.parametrize("n,tile_pairs,half", [(60_001, 1, 8.0), (60_001, 1, 1.0), (400_000, 3, 8.0), (49_153, 1, 200.0)])
def test_order_of_the_loads_changes_nothing(nb, n, tile_pairs, half):
    def bunch(m, seed):
        b = H.DeviceBunch(m)
        b.generate(seed, W.SIGMA_Z, W.SIGMA_E)
        return b

    def options():
        return H.TrackingOptions(seed=9, monitor=True, tile_pairs=tile_pairs, charge=2e-9,
                                 resonators=[W.RESONATOR_BB], bin_half_width_sigmas=half)

    def params(excitation):
        return H.SimulationParameters.from_dict(W.ring_3gev_lattice(4, flags=(True,) * 4 + (excitation,)))
    alone, beside, other = bunch(n, 5), bunch(n, 5), bunch(1000, 6)
    r = alone.evolve(params(True), nb, options())
    rs = H.batch_evolve([beside, other], [nb, 64], [params(True), params(False)], [options(), options()])
    for a, g in zip(alone.download(), beside.download()):
        assert np.array_equal(a, g)
    assert np.array_equal(r.monitor, rs[0].monitor) and r.E0 == rs[0].E0
    for b in (alone, beside, other):
        b.close()
