"""Device memory of served jobs: taken at admission, where a job that does not fit
fails alone, and within the server's budget."""
import pytest
import torch

from helpers import W

import haissinskijulia_amd as H

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _job(n, nbins, turns, **options):
    return H.Job(params=H.SimulationParameters.from_dict(W.ring_3gev_lattice(turns)), n=n, nbins=nbins,
                 particle_seed=3, sigma_z=W.SIGMA_Z, sigma_E=W.SIGMA_E,
                 options=H.TrackingOptions(seed=5, charge=1e-9, resonators=[W.RESONATOR_BB], **options))


@pytest.mark.parametrize("n,nbins", [(1_000_000, 65536), (10_000_000, 131072)])
def test_a_jobs_buffers_are_taken_at_admission(n, nbins):
    # 256 slabs of 98304 bytes are 25 MB; a turn's launch tables stay below 2.  A
    # job before: the runtime allocates for a process's first launches (16 MB)
    srv = H.Server(budget_bytes=8 << 30, max_slots=4)
    srv.submit(_job(n, nbins, 3))
    srv.run(10)
    job = srv.submit(_job(n, nbins, 3))
    srv.tick(0)
    admitted = _free()
    srv.tick(1)
    assert admitted - _free() <= 4 * MB
    res = {r.job_id: r for r in srv.run(10)}
    srv.close()
    assert res[job].status == 0


@pytest.mark.parametrize("n,nbins,options", [(524_288, 65536, dict(tile_pairs=1)), (40_000, 131072, {}),
                                             (200_000, 5000, dict(tile_pairs=1))])
def test_admitted_jobs_stay_within_the_budget(n, nbins, options):
    # 64 MiB; launch tables, and what the runtime rounds sizes up to, 8
    srv = H.Server(budget_bytes=64 * MB, max_slots=32)
    srv.submit(_job(n, nbins, 2, **options))
    srv.run(10)
    before = _free()
    jobs = [srv.submit(_job(n, nbins, 4, **options)) for _ in range(12)]
    most, left = 0, 1
    while left:
        left = srv.tick(1)
        most = max(most, before - _free())
        print(f"{left} jobs left, {most / MB:.1f} MiB at most", flush=True)
    assert most <= 72 * MB
    assert all(r.status == 0 for r in srv.poll()) and len(jobs) == 12
    srv.close()
