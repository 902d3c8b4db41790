"""32-bit counts of a whole histogram in LDS, its window of 16-bit counts, and counts
in global memory, at the sizes where one takes over from the other.

Tiles of 32 chunks (32768 pairs) never take the window.  The bunches are those of
test_gpu_hist_window.py, whose sums are exact in any order, so that every form
gives the same bits."""
import numpy as np
import pytest

from helpers import W
from test_gpu_hist_window import _gaussian, _same

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [34560, 34561, 34562, 40001, 40700, 40701, 40702])
@pytest.mark.parametrize("n", [49_152, 49_153, 2_499_998, 2_499_999])
def test_forms_agree(nb, n):
    _same(_gaussian(n), nb, 0, 2.5, (True, True, False, True, True))


@pytest.mark.parametrize("nb", [34561, 40700, 40701])
@pytest.mark.parametrize("other,other_turns", [(2_400_001, 3), (2_400_001, 1), (20_000, 2)])
def test_a_bunch_changes_its_form_with_the_batch(nb, other, other_turns):
    # alone by 32 bits; beside the larger bunch by the window, until that retires
    def bunch(n, seed):
        b = H.DeviceBunch(n)
        b.generate(seed, 4e-3, 3e6)
        return b

    def params(turns):
        return H.SimulationParameters.from_dict(W.ring_3gev_lattice(turns))

    def options():
        return H.TrackingOptions(seed=9, monitor=True, charge=2e-9, resonators=[W.RESONATOR_BB])
    alone, beside, big = bunch(120_001, 5), bunch(120_001, 5), bunch(other, 6)
    r = alone.evolve(params(4), nb, options())
    rs = H.batch_evolve([beside, big], [nb, 40000], [params(4), params(other_turns)], [options(), options()])
    for a, g in zip(alone.download(), beside.download()):
        assert np.array_equal(a, g)
    assert np.array_equal(r.monitor, rs[0].monitor) and r.E0 == rs[0].E0
    for b in (alone, beside, big):
        b.close()
