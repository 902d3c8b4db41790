"""Calls on host arrays, whose small copies go through one kernel, and results of
many bunches fetched together: the same bits as resident bunches one by one."""
import numpy as np
import pytest

from helpers import W
from oracle import oracle as O

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


def _resident(z0, e0, p, nb, seed):
    b = H.DeviceBunch(z0.size)
    b.upload(z0, e0)
    r = b.evolve(p, nb, H.TrackingOptions(seed=seed))
    out = (*b.download(), r.sigma_E, r.sigma_z, r.E0)
    b.close()
    return out


@pytest.mark.parametrize("n", [1, 2, 3, 1023, 32767, 32768, 32769, 70_001])   # 256 KB an array: 32768
def test_host_call_equals_resident(n):
    z0, e0 = O.generate_gaussian(5, 0.0, 4e-3, 0.0, 1e6, n)
    p = H.SimulationParameters.from_dict(W.reference_benchmark_lattice(3))
    nb = 64
    ref = _resident(z0, e0, p, nb, 7)
    part = H.Particles(z0.copy(), e0.copy())
    got = H.longitudinal_evolve(part, p, H.create_simulation_buffers(n, nb), H.MI355X.default(), True, H.TrackingOptions(seed=7))
    assert np.array_equal(part.coordinates.z, ref[0], equal_nan=True)
    assert np.array_equal(part.coordinates.dE, ref[1], equal_nan=True)
    assert np.array_equal(got, ref[2:], equal_nan=True)


def test_results_of_many_bunches():
    p = H.SimulationParameters.from_dict(W.reference_benchmark_lattice(3))
    sizes = [500 + 37 * k for k in range(70)]
    parts = [O.generate_gaussian(k, 0.0, 4e-3, 0.0, 1e6, n) for k, n in enumerate(sizes)]
    bunches = [H.DeviceBunch(n) for n in sizes]
    for b, (z, e) in zip(bunches, parts):
        b.upload(z, e)
    rs = H.batch_evolve(bunches, [64] * 70, [p] * 70, [H.TrackingOptions(seed=k) for k in range(70)])
    for k, (b, r, (z, e)) in enumerate(zip(bunches, rs, parts)):
        ref = _resident(z, e, p, 64, k)
        zg, eg = b.download()
        assert np.array_equal(zg, ref[0]) and np.array_equal(eg, ref[1])
        assert (r.sigma_E, r.sigma_z, r.E0) == ref[2:]
        b.close()
