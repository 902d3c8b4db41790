"""The bin phase of grids with 64-bin blocks (k_bin_64) against a launch per
phase, bit for bit: ragged last blocks, one to four reduction slices, a wake
over part of the grid, and turns in which no particle is binned."""
import numpy as np
import pytest

from helpers import W
from oracle import oracle as O

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


def _both(z0, e0, nbins, flags, lag, turns=20):
    p = H.SimulationParameters.from_dict(W.ring_3gev_lattice(n_turns=turns, flags=flags))
    kw = dict(resonators=[W.RESONATOR_BB], charge=2e-9) if lag else {}
    outs = []
    for bw in (0, -1):
        b = H.DeviceBunch(z0.size)
        b.upload(z0, e0)
        r = b.evolve(p, nbins, H.TrackingOptions(seed=3, bin_half_width_sigmas=4.0, monitor=True,
                                                 bin_whole=bw, fft_block=64, tile_pairs=1, **kw))
        outs.append((*b.download(), r))
        b.close()
    (za, ea, ra), (zb, eb, rb) = outs
    np.testing.assert_array_equal(za, zb)
    np.testing.assert_array_equal(ea, eb)
    assert (ra.sigma_E, ra.sigma_z, ra.E0) == (rb.sigma_E, rb.sigma_z, rb.E0)
    np.testing.assert_array_equal(ra.monitor, rb.monitor)
    return ra


@pytest.mark.parametrize("n,nbins,flags,lag", [
    (5_000, 65, (True, True, True, True, True), True),        # two blocks, one bin in the second
    (5_001, 127, (True, True, True, True, True), False),      # the reference's wake and current
    (9_000, 192, (True, False, True, True, True), True),      # an odd number of blocks
    (9_000, 320, (True, True, False, True, True), True),      # no E0 update, five blocks
    (20_000, 961, (True, True, True, True, True), True),      # sixteen blocks, one bin in the last
    (20_000, 1023, (True, True, True, True, True), False),
    (131_073, 1024, (True, True, True, True, True), True),    # two reduction slices
    (300_001, 1000, (True, True, True, True, True), False),   # three
    (500_001, 1024, (True, True, True, True, True), True),    # four
])
def test_64_bin_blocks_equal_the_launches(n, nbins, flags, lag):
    z0, e0 = O.generate_gaussian(31, 0.0, 4e-3, 0.0, 3e6, n)
    r = _both(z0, e0, nbins, flags, lag)
    assert 0 < r.monitor[-1, 3] <= n


def test_64_bin_blocks_with_no_particle_binned():
    # no spread: the grid is +-1 um around 0, the bunch at 10 mm
    r = _both(np.full(3_000, 0.01), np.zeros(3_000), 256, (True, True, True, True, False), True, turns=3)
    assert np.all(r.monitor[:, 3] == 0)
