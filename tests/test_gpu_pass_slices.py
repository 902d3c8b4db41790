"""The turn pass with its tiles split over two workgroups.

Where the batch has few tiles, two workgroups of half the waves each take a
tile.  A tile's sums are per wave, so a bunch alone (split) and beside one that
fills the chip (not split) gets the same bits: at the edges of chunks and tiles,
with the deposit, with a partial window of P and with the windowed histogram."""
import numpy as np
import pytest

from helpers import W

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,update_E0", [(100, True), (100, False), (16384, True), (40001, True)])
@pytest.mark.parametrize("n,tile_pairs", [(1, 1), (2, 1), (3, 1), (1023, 1), (1025, 1), (2049, 1), (6145, 3),
                                          (262_143, 0), (262_144, 0)])
def test_split_tiles(nb, update_E0, n, tile_pairs):
    p = H.SimulationParameters.from_dict(W.ring_3gev_lattice(3, flags=(True, True, update_E0, True, True)))

    def bunch(n, seed):
        b = H.DeviceBunch(n)
        b.generate(seed, 4e-3, 3e6)
        return b

    def options(tile_pairs):
        return H.TrackingOptions(seed=9, tile_pairs=tile_pairs, monitor=True, charge=2e-9,
                                 resonators=[W.RESONATOR_BB])
    alone, beside, big = bunch(n, 5), bunch(n, 5), bunch(600_000, 6)
    r = alone.evolve(p, nb, options(tile_pairs))
    rs = H.batch_evolve([beside, big], [nb, 1024], [p, p], [options(tile_pairs), options(1)])
    for a, g in zip(alone.download(), beside.download()):
        assert np.array_equal(a, g)
    assert np.array_equal(r.monitor, rs[0].monitor, equal_nan=True) and r.E0 == rs[0].E0
    for b in (alone, beside, big):
        b.close()
