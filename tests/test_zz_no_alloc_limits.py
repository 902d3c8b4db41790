"""The largest bunches of hm_evolve_device_noalloc.

Its work buffers share one scratch array, so tiles of 1024 pairs (672 bytes of
sums each) bound a bunch's particles by what the tables of its bins leave.  The
sizes are those that filled 8 MiB with packed counters (8 B per bin of
histogram, 20 B of deposit) and with one entry of 16 bytes per tile of launch
tables: they have to be taken, and give the bits of the allocating call."""
import ctypes as C

import numpy as np
import pytest

from helpers import W

import haissinskijulia_amd as H
from haissinskijulia_amd import _lib

pytestmark = pytest.mark.gpu

ALL_ON = (True,) * 5


@pytest.mark.parametrize("n,nbins,flags", [
    (24_930_000, 0, (False, True, False, True, True)), (24_930_000, 0, (False, True, True, True, True)),
    (24_800_000, 256, ALL_ON), (22_920_000, 4096, ALL_ON), (22_280_000, 5814, ALL_ON), (17_890_000, 16384, ALL_ON),
    (10_870_000, 32768, ALL_ON), (10_870_000, 32768, (True, True, False, True, True))])
def test_largest_bunches_of_small_tiles(n, nbins, flags):
    L = _lib.load()
    p = H.SimulationParameters.from_dict(W.ring_3gev_lattice(1, flags=flags))

    def options():
        return H.TrackingOptions(seed=3, tile_pairs=1, charge=1e-9, resonators=[W.RESONATOR_BB])
    a, b = H.DeviceBunch(n), H.DeviceBunch(n)
    for x in (a, b):
        x.generate(7, W.SIGMA_Z, W.SIGMA_E)
    zp, ep, keep, r = C.c_void_p(), C.c_void_p(), [], _lib.HmResult()
    _lib.check(L.hm_bunch_device_ptrs(a._h, C.byref(zp), C.byref(ep)))
    o = options()._c(keep, n, 1, nbins)
    _lib.check(L.hm_evolve_device_noalloc(a.device.ctx, zp, ep, n, nbins, C.byref(p._c()), C.byref(o), C.byref(r)))
    rb = b.evolve(p, nbins, options())
    assert (r.sigma_E, r.sigma_z, r.E0) == (rb.sigma_E, rb.sigma_z, rb.E0)
    for x, y in zip(a.download(), b.download()):
        assert np.array_equal(x, y)
    a.close()
    b.close()
