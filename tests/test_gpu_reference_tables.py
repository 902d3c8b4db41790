"""The reference's wake and delta tables, made on the device from the bin centres.

One turn with the wake alone leaves P at each particle: compared with the
oracle's tables and its FFT convolution, for numbers of bins around and off the
powers of two (the centre's quotient is inexact), a grid of the smallest width,
and one so wide that the wake underflows within it.  Particles beyond the end
centres are left out: clamped to the last one, their weight is 0 or 1 by the
last place of sigma_z, which the oracle need not share."""
import numpy as np
import pytest

from helpers import POTENTIAL_RTOL, W, normwise
from oracle import oracle as O

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [1, 2, 3, 5, 64, 100, 1023, 1024, 1025, 4099, 40001])
@pytest.mark.parametrize("half,delta_sigma", [(7.5, 0.0), (3.0, 0.01), (2000.0, 0.0), (1e-8, -1.0)])
def test_reference_tables(nb, half, delta_sigma):
    n = 20_001
    z0, e0 = O.generate_gaussian(5, 0.0, 4e-3, 0.0, 1e6, n)
    p = W.reference_benchmark_lattice(1, (True, False, False, False, False))
    zr, er, _ = O.evolve(z0, e0, nb, p, seed=3, delta_sigma=delta_sigma, bin_half_width_sigmas=half)
    _, en, _ = O.evolve(z0, e0, 0, W.reference_benchmark_lattice(1, (False,) * 5), seed=3)
    b = H.DeviceBunch(n)
    b.upload(z0, e0)
    r = b.evolve(H.SimulationParameters.from_dict(p), nb,
             H.TrackingOptions(seed=3, delta_sigma=delta_sigma, bin_half_width_sigmas=half))
    z, e = b.download()
    b.close()
    assert normwise(z, zr) <= 1e-14
    # the kicks, to the oracle's convolution and the rounding of dE they are taken from
    inside = np.abs(z) < r.bin_half_width * (1 - 1 / nb) if nb > 1 else slice(None)
    kick, ref = (en - e)[inside], (en - er)[inside]
    if not ref.size:
        return
    scale = np.sqrt(np.mean(ref * ref))
    assert np.max(np.abs(kick - ref)) <= POTENTIAL_RTOL * scale + 2 ** -52 * np.max(np.abs(en[inside]))
