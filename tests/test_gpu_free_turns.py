"""Turns without a wake and without the E0 update, many per launch
(k_free_turns), against one pass per turn (which `timing` asks for): the same
expressions, so the same bits."""
import numpy as np
import pytest

from helpers import W
from oracle import oracle as O

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags", [(False, True, False, True, True), (False, False, False, True, True),
                                   (False, True, False, False, True), (False, True, False, True, False)])
@pytest.mark.parametrize("n", [1, 2, 3, 511, 512, 513, 2049, 70_001])
def test_free_turns_equal_one_pass_per_turn(n, flags):
    z0, e0 = O.generate_gaussian(8, 0.0, 4e-3, 0.0, 3e6, n)
    p = H.SimulationParameters.from_dict(W.ring_3gev_lattice(13, flags=flags))
    for normals in (None, np.vstack([O.normals(4, t, 0, n) for t in range(13)])):
        outs = []
        for timing in (False, True):
            b = H.DeviceBunch(n)
            b.upload(z0, e0)
            r = b.evolve(p, 0, H.TrackingOptions(seed=21, turn_offset=5, monitor=True, timing=timing,
                                                 normals=normals))
            outs.append((*b.download(), r))
            b.close()
        (za, ea, ra), (zb, eb, rb) = outs
        np.testing.assert_array_equal(za, zb)
        np.testing.assert_array_equal(ea, eb)
        np.testing.assert_array_equal(ra.monitor, rb.monitor)
        assert (ra.sigma_E, ra.sigma_z, ra.E0, ra.turns_done, ra.drift_skipped) == \
               (rb.sigma_E, rb.sigma_z, rb.E0, rb.turns_done, rb.drift_skipped)


def test_free_turns_in_batches_and_ticks():
    """Uneven turn counts in a batch, the same with a wake bunch beside them
    (one pass per turn for all), and a server's ticks: the bits of each alone."""
    free = (False, True, False, True, True)
    sizes, turns = (4_001, 30_000, 513), (20, 7, 33)
    kw = dict(sigma_z=W.SIGMA_Z, sigma_E=W.SIGMA_E)

    def lattice(t, flags=free):
        return H.SimulationParameters.from_dict(W.ring_3gev_lattice(t, flags=flags))

    def bunches(k):
        bs = [H.DeviceBunch(n) for n in sizes[:k]]
        for i, b in enumerate(bs):
            b.generate(50 + i, **kw)
        return bs

    opts = [H.TrackingOptions(seed=60 + i) for i in range(3)]
    alone = []
    for i, b in enumerate(bunches(3)):
        r = b.evolve(lattice(turns[i]), 0, opts[i])
        alone.append((*b.download(), r.sigma_E, r.sigma_z, r.E0, r.turns_done))
    for wake in (False, True):
        bs = bunches(3)
        nb, ps, os_ = [0] * 3, [lattice(t) for t in turns], list(opts)
        if wake:
            w = H.DeviceBunch(9_000)
            w.generate(70, **kw)
            bs, nb, ps = bs + [w], nb + [256], ps + [lattice(25, (True,) * 5)]
            os_.append(H.TrackingOptions(seed=70, resonators=[W.RESONATOR_BB], charge=1e-9))
        rs = H.batch_evolve(bs, nb, ps, os_)
        for (za, ea, *ra), b, r in zip(alone, bs, rs):
            z, e = b.download()
            np.testing.assert_array_equal(z, za)
            np.testing.assert_array_equal(e, ea)
            assert [r.sigma_E, r.sigma_z, r.E0, r.turns_done] == ra
    srv = H.Server(1 << 30, 4)
    ids = [srv.submit(H.Job(params=lattice(turns[i]), n=sizes[i], nbins=0, particle_seed=50 + i,
                            options=opts[i], **kw)) for i in range(3)]
    done = {r.job_id: r.result for r in srv.run(6)}
    srv.close()
    for i, (_, _, *ra) in zip(ids, alone):
        r = done[i]
        assert [r.sigma_E, r.sigma_z, r.E0, r.turns_done] == ra
