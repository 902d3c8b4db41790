"""The turn's sigma_z (evolution.jl:357) without contraction.

Multiplies and adds of the per-particle path round separately, the squares of z
in the pass's sums among them.  Bunches of a few particles, whose sums have one
order: the turn monitor's centroid and sigma_z are, to the last bit, those of
compute_global_std's expressions (utils.jl:589-605) in numpy on the same z."""
import numpy as np
import pytest

from helpers import W

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


def _sums(x):
    """Thread 0 adds its pair, then the odd last particle; thread 1 its pair."""
    first = x[0] + x[1]
    if x.size % 2:
        first = first + x[-1]
    return first + (x[2] + x[3]) if x.size > 3 else first


@pytest.mark.parametrize("flags", [(True,) * 5, (True, False, False, False, False)])
@pytest.mark.parametrize("n", [2, 3, 4, 5])
def test_sigma_z_rounds_each_square(n, flags):
    p = H.SimulationParameters.from_dict(W.ring_3gev_lattice(1, flags=flags))
    for seed in range(40):
        b = H.DeviceBunch(n)
        b.generate(seed, W.SIGMA_Z, W.SIGMA_E)
        r = b.evolve(p, 64, H.TrackingOptions(seed=seed, monitor=True, charge=1e-9, resonators=[W.RESONATOR_BB]))
        z, _ = b.download()
        b.close()
        mean = _sums(z) / n
        var = _sums(z * z) / n - mean * mean
        assert r.monitor[0, 0] == mean
        assert r.monitor[0, 1] == np.sqrt(max(0.0, var * n / (n - 1)))
