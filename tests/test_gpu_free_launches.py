"""Turns without a wake and without the E0 update over more than one launch: the bits
of one launch of the pass per turn (which timing asks for)."""
import numpy as np
import pytest

from helpers import W

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


def test_more_turns_than_a_launch_takes():
    turns = 50_003   # a launch of a small bunch takes 50000
    p = H.SimulationParameters.from_dict(W.ring_3gev_lattice(turns, flags=(False, True, False, True, True)))
    out = []
    for timing in (False, True):
        b = H.DeviceBunch(257)
        b.generate(5, W.SIGMA_Z, W.SIGMA_E)
        r = b.evolve(p, 0, H.TrackingOptions(seed=9, monitor=True, timing=timing))
        out.append((*b.download(), r.monitor, r.turns_done))
        b.close()
    for a, g in zip(*out):
        assert np.array_equal(a, g)


@pytest.mark.parametrize("n,turns", [(4_194_304, 3), (4_194_306, 1), (4_200_001, 3), (4_197_377, 2), (67_110_913, 1)])
def test_several_pairs_per_thread(n, turns):
    # four pairs per thread from 4194306 particles on, sixteen from 67108866; odd sizes, a last
    # item of one particle (4197377 = 4096 * 1024 + 3 * 1024 + 1)
    p = H.SimulationParameters.from_dict(W.ring_3gev_lattice(turns, flags=(False, True, False, True, True)))
    out = []
    for timing in (False, True):
        b = H.DeviceBunch(n)
        b.generate(5, W.SIGMA_Z, W.SIGMA_E)
        r = b.evolve(p, 0, H.TrackingOptions(seed=9, timing=timing, tile_pairs=64))
        out.append((*b.download(), r.sigma_E, r.sigma_z, r.E0))
        b.close()
    for a, g in zip(*out):
        assert np.array_equal(a, g)
