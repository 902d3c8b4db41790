"""The turn pass at the edges of its tiles against the oracle's stages.

The pass walks a tile in chunks of 1024 pairs, prefetching the next chunk (the
next tile's first at a tile's end); only a bunch's last chunk may be short, its
idle lanes re-reading the last pair.  Sizes around one chunk, one tile and the
single particle of an odd bunch, for one and three chunks per tile.  The counts
and the potential are the oracle's for the device's own positions and grid, so a
particle at a bin edge cannot fall on two sides of it."""
import numpy as np
import pytest

from helpers import COORD_RTOL, W, normwise
from oracle import oracle as O

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu

NB, CHARGE, HALF = 100, 2e-9, 2.5   # bins over +-2.5 sigma: some particles are off the grid


def _device(z0, e0, p, tile_pairs):
    b = H.DeviceBunch(z0.size)
    b.upload(z0, e0)
    r = b.evolve(H.SimulationParameters.from_dict(p), NB,
                 H.TrackingOptions(seed=9, tile_pairs=tile_pairs, monitor=True, charge=CHARGE,
                                   resonators=[W.RESONATOR_BB], bin_half_width_sigmas=HALF))
    z, e = b.download()
    b.close()
    return z, e, r


@pytest.mark.parametrize("update_E0", [True, False])   # the all-flags pass with the deposit, the generic one
@pytest.mark.parametrize("n,tile_pairs", [(2, 1), (3, 1), (2047, 1), (2048, 1), (2049, 1), (2050, 1),
                                          (4095, 1), (4097, 1), (6143, 3), (6144, 3), (6145, 3),
                                          (6147, 3), (12289, 3), (14337, 3)])
def test_pass_at_tile_edges(n, tile_pairs, update_E0):
    z0, e0 = O.generate_gaussian(5, 0.0, 4e-3, 0.0, 3e6, n)
    flags = (True, True, update_E0, True, True)
    free = (False, True, False, True, True)
    p = W.ring_3gev_lattice(1, flags=flags)
    z1, e1, r1 = _device(z0, e0, p, tile_pairs)
    # the turn without the wake, then the wake of the device's own positions
    zr, er, rr = O.evolve(z0, e0, 0, W.ring_3gev_lattice(1, flags=free), seed=9)
    assert rr.status == 0 and normwise(z1, zr) <= COORD_RTOL
    edges, centers, step = O.bin_grid(r1.bin_half_width, NB)
    assert r1.bin_half_width == pytest.approx(HALF * O.global_std(z0), rel=1e-13)
    counts = O.histogram(z1, edges[0], edges[-1], 1.0 / step, NB)
    assert r1.monitor[0, 3] == counts.sum()
    wake = np.array([O.resonator_wake(k * step, *W.RESONATOR_BB) for k in range(NB)])
    g = counts / max(counts.sum(), 1)
    P = CHARGE * np.array([np.dot(wake[:NB - k], g[k:]) for k in range(NB)])
    er = er - O.interpolate(z1, centers, P)
    E0 = p["E0"]
    if update_E0:
        m = np.mean(er - e0)
        E0 += m
        er = er - m
    assert normwise(e1, er) <= COORD_RTOL
    assert r1.E0 == pytest.approx(E0, rel=1e-14)
    # the next turn of one call starts with that kick: as a turn of its own
    # from the kicked bunch, its normals scaled from one call's sigma_E0 to the other's
    z2, _, _ = _device(z0, e0, dict(p, n_turns=2), tile_pairs)
    normals = O.normals(9, 1, 0, n)[None, :] * (O.global_std(e0) / O.global_std(e1))
    zr, _, rr = O.evolve(z1, e1, 0, dict(W.ring_3gev_lattice(1, flags=free), E0=r1.E0), normals=normals)
    assert rr.status == 0 and normwise(z2, zr) <= COORD_RTOL
