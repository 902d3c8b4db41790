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
