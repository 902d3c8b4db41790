"""The reference's wake and delta tables where the whole bunch lies on the grid.

test_gpu_reference_tables.py tracks a 4 mm bunch; on its narrowest grid (+-1e-6 m,
the least width) none of the particles that it compares is left.  Here the
particles lie within that grid, so P of nearly every bin is met, with the reference's
kernel width, one as narrow as the grid, and none (a constant lambda, also on a
grid of ordinary width).  Compared as there: one turn with the wake alone, the
kicks against the oracle's to its convolution and the rounding of dE."""
import numpy as np
import pytest

from helpers import POTENTIAL_RTOL, W
from oracle import oracle as O

import haissinskijulia_amd as H

N = 20_001
BINS = [2, 3, 5, 64, 100, 1023, 1024, 1025, 4099, 40001]
GRIDS = {"least": (1e-6, 100.0, 1e-4), "narrow": (1e-6, 100.0, 3.0), "ordinary": (8e-3, 1e6, 3.0)}


def _bunch(grid):
    width, sigma_E, half = GRIDS[grid]
    rng = np.random.default_rng(11)
    return rng.uniform(-width, width, N), rng.normal(0.0, sigma_E, N), half


def _oracle(grid, nb, delta_sigma):
    z, e, half = _bunch(grid)
    p = W.reference_benchmark_lattice(1, (True, False, False, False, False))
    zr, er, _ = O.evolve(z, e, nb, p, seed=3, delta_sigma=delta_sigma, bin_half_width_sigmas=half)
    zn, en, _ = O.evolve(z, e, 0, W.reference_benchmark_lattice(1, (False,) * 5), seed=3)
    return zr, er, en


def _close(kick, ref, en):
    scale = np.sqrt(np.mean(ref * ref))
    return np.max(np.abs(kick - ref)) <= POTENTIAL_RTOL * scale + 2 ** -52 * np.max(np.abs(en))


def _inside(z, half_width, nb):
    keep = np.abs(z) < half_width * (1 - 1 / nb)
    assert keep.sum() >= (N // 3 if nb == 2 else N // 2)
    return keep


@pytest.mark.gpu
@pytest.mark.parametrize("nb", BINS)
@pytest.mark.parametrize("grid,delta_sigma", [("least", 0.0), ("least", 4e-7), ("least", -1.0), ("narrow", 4e-7),
                                              ("narrow", -1.0), ("ordinary", 0.0), ("ordinary", -1.0)])
def test_kicks_on_the_grid(nb, grid, delta_sigma):
    zr, er, en = _oracle(grid, nb, delta_sigma)
    z0, e0, half = _bunch(grid)
    b = H.DeviceBunch(N)
    b.upload(z0, e0)
    p = W.reference_benchmark_lattice(1, (True, False, False, False, False))
    r = b.evolve(H.SimulationParameters.from_dict(p), nb,
                 H.TrackingOptions(seed=3, delta_sigma=delta_sigma, bin_half_width_sigmas=half))
    z, e = b.download()
    b.close()
    # z up to its own last place: the device multiplies by 1 / rf where the oracle divides.  A last
    # place of the phase, 1.6e-16 m, would be 1e-10 of the least grid
    same = np.abs(z - zr) <= 2 ** -51 * np.abs(z)
    assert same.sum() >= 0.99 * N
    keep = _inside(z, r.bin_half_width, nb) & same
    assert _close((en - e)[keep], (en - er)[keep], en[keep])


@pytest.mark.parametrize("grid", sorted(GRIDS))
def test_a_wrong_table_would_be_seen(grid):
    """The comparison itself: the oracle's own kicks with a kernel narrower by 1e-6."""
    z, er, en = _oracle(grid, 100, 0.15)
    _, ew, _ = _oracle(grid, 100, 0.15 * (1 - 1e-6))
    _, _, half = _bunch(grid)
    keep = np.abs(z) < np.abs(z).max() / 2
    assert keep.sum() > N // 4
    assert not _close((en - ew)[keep], (en - er)[keep], en[keep])
