"""Histograms of more bins than the LDS holds: the window of 16-bit counts.

Tiles of 32 chunks (32768 pairs) exceed what a 16-bit count can hold, so they
take the path that adds every particle to global memory; smaller tiles take the
window.  The counts are whole numbers, and the bunches start on a lattice with
mean zero, so that the sums behind their sigmas are exact in any order: without
the energy update (the only other sum over tiles that reaches the particles), or
with one tile, both paths give the same bits.  Sizes around the window's own, an odd number of bins, particles
off the grid, workgroups with several runs, a bin with a whole run's particles."""
import numpy as np
import pytest

from helpers import W

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


def _run(bunch, nb, tile_pairs, half, flags, turns=3):
    p = W.ring_3gev_lattice(turns, flags=flags)
    r = bunch.evolve(H.SimulationParameters.from_dict(p), nb,
                     H.TrackingOptions(seed=9, tile_pairs=tile_pairs, monitor=True, charge=2e-9,
                                       resonators=[W.RESONATOR_BB], bin_half_width_sigmas=half))
    z, e = bunch.download()
    return z, e, r.monitor[:, 3], r.E0


def _same(make, nb, tile_pairs, half, flags):
    out = []
    for tp in (tile_pairs, 32):
        b = make()
        out.append(_run(b, nb, tp, half, flags))
        b.close()
    for a, g in zip(*out):
        assert np.array_equal(a, g)
    return out[0]


def _gaussian(n):
    rng = np.random.default_rng(5)
    half = np.rint(rng.standard_normal((2, n // 2)) * [[262], [732]])   # of 2^-16 m and 4096 eV
    x = np.concatenate([half, np.zeros((2, n % 2)), -half], axis=1)

    def make():
        b = H.DeviceBunch(n)
        b.upload(x[0] * 2.0 ** -16, x[1] * 4096.0)
        return b
    return make


@pytest.mark.parametrize("nb", [33500, 34001, 40001, 49151, 49152, 49153, 49154, 65536, 131072])
@pytest.mark.parametrize("n,tile_pairs,update_E0", [(50001, 31, True), (50001, 31, False), (200_003, 1, False),
                                                    (1, 1, False)])
def test_window_counts(nb, n, tile_pairs, update_E0):
    _same(_gaussian(n), nb, tile_pairs, 2.5, (True, True, update_E0, True, True))


def test_several_runs_per_workgroup():
    _, _, counts, _ = _same(_gaussian(17_000_001), 131072, 31, 7.5, (True, True, False, True, True))
    assert counts[0] > 16_900_000


def test_one_bin_holds_a_run():
    z0 = np.zeros(63488)
    z0[:4] = [-0.3, 0.3, -0.01, 0.01]

    def make():
        b = H.DeviceBunch(z0.size)
        b.upload(z0, np.zeros(z0.size))
        return b
    _same(make, 65536, 31, 7.5, (True, True, False, False, False))
