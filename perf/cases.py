"""The tracking work that this library is used for, as timed cases.

A case is one call of a user's program: a bunch already in hand (on the host,
or resident in HBM) is tracked for a number of turns and its coordinates and
spreads come back.  A repeated call goes on with the bunch where the last one
left it, from the next turn of the random stream, at the lattice's nominal
energy.  Lattices, wakes, bin counts and bunch shapes are those of
``haissinskijulia_amd.workloads``, the integration benchmark
(``haissinskijulia_amd.benchlog``), ``bench.py`` and the equilibrium tests.

Kinds of case:

* ``host``     ``longitudinal_evolve`` on NumPy arrays, the reference's call;
* ``resident`` ``DeviceBunch.evolve``;
* ``batch``    ``batch_evolve`` over several uneven bunches;
* ``serve``    jobs through ``Server`` until all of them are done.

``exact`` is the same tracking in plain torch, one reference stage after the
other in FP64.
"""
import math
import random

import numpy as np
import torch

import haissinskijulia_amd as H
from haissinskijulia_amd import workloads as W

C_LIGHT = W.SPEED_LIGHT
TWO_PI = 2 * math.pi
ALL_ON = "wake,eta,E0,SR,QE"


def _resident(name, n, nbins, turns, **kw):
    c = dict(kind="resident", n=n, nbins=nbins, turns=turns, lattice="ring3", charge_nC=1.0, resonators=1,
             half_width=8.0, flags=ALL_ON, monitor=False)
    c.update(kw)
    return dict(c, name=name) if name else c


def _reference(name, kind, n, turns, **kw):
    """The integration benchmark's own shape: its lattice, its wake and its N/100 bins."""
    return _resident(name, n, H.next_power_of_two(max(64, round(n / 100))), turns, kind=kind, lattice="reference",
                     charge_nC=0.0, resonators=0, half_width=7.5, **kw)


def listed():
    return [
        # a first try of the drop-in call: a few thousand particles, a few turns
        _reference("host_4e3", "host", 4097, 10),
        # the drop-in call at the smallest size of the integration benchmark
        _reference("host_1e5", "host", 100_000, 100),
        # one member of an equilibrium ensemble: small, many turns, watched turn by turn
        _resident("ensemble_2e4", 20_000, 512, 1000, monitor=True),
        # the small tracking workload
        _resident("ring3_1e5", 100_000, 1024, 1000, half_width=6.0),
        # the integration benchmark's middle and largest sizes (the largest has
        # more bins than fit a histogram in LDS)
        _reference("reference_1e6", "resident", 1_000_000, 100),
        _reference("reference_1e7", "resident", 10_000_000, 50),
        # towards the equilibrium at fixed energy and slippage: few bins, no E0 update
        _resident("equilibrium_1e6", 1_000_000, 512, 300, flags="wake,SR,QE", monitor=True),
        # tracking without a wake, an odd number of particles
        _resident("nowake_3e6", 3_000_001, 0, 200, flags="eta,SR,QE", charge_nC=0.0, resonators=0),
        # the two large tracking workloads
        _resident("ring3_1e7", 10_000_000, 8192, 200, charge_nC=5.0),
        _resident("ring3_1e8", 100_000_000, 16384, 100, charge_nC=10.0, resonators=2),
        # a parameter scan: uneven bunches advanced together
        dict(name="scan_28", kind="batch", count=28, n_lo=10_000, n_hi=4_000_000, nbins=4096, turns=200, sizes=3),
        # served jobs, a fifth of them finite-difference pairs
        dict(name="serve_24", kind="serve", count=24, n_lo=10_000, n_hi=1_000_000, nbins=1024, turns_lo=100,
             turns_hi=500, per_tick=100, sizes=5),
    ]


def _charge(rng, turns):
    """Charge in nC.  Beyond about 3 nC this ring's bunch is above its microwave threshold: over several hundred turns
    any rounding grows until two correct trackings differ, so the longer runs are those of the stable bunches."""
    return round(rng.uniform(0.5, 10.0 if turns <= 200 else 2.5), 3)


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("resident", "host", "batch", "serve"), (11, 3, 3, 3))[0]
    if kind == "resident":
        n = _log_int(rng, 4e3, 1e8)
        turns = min(_log_int(rng, 10, 1000), max(10, int(4e9 / n)))
        if rng.random() < 0.25 and n <= 10_000_000:
            return _reference(None, "resident", n, min(turns, 200))
        flags = rng.choices((ALL_ON, "wake,SR,QE", "wake,eta,SR,QE", "eta,SR,QE", "eta,E0,SR"), (12, 2, 2, 2, 1))[0]
        wake = "wake" in flags
        near = 2 ** max(8, min(14, round(math.log2(n / 100) + rng.uniform(-1, 1))))
        nbins = near if rng.random() < 0.8 else int(near * rng.uniform(0.6, 1.0))
        return _resident(None, n, nbins if wake else 0, turns, charge_nC=_charge(rng, turns) if wake else 0.0,
                         resonators=rng.choice((1, 1, 2)) if wake else 0, half_width=rng.choice((6.0, 8.0)),
                         flags=flags, monitor=wake and rng.random() < 0.25)
    if kind == "host":
        return _reference(None, "host", _log_int(rng, 2e3, 2e6), rng.choice((10, 30, 100)))
    n_lo = _log_int(rng, 8e3, 3e4)
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(6, 28), n_lo=n_lo, n_hi=_log_int(rng, 2e5, 4e6),
                    nbins=rng.choice((1024, 2048, 4096)), turns=_log_int(rng, 30, 200), sizes=rng.randrange(1000))
    return dict(kind="serve", count=rng.randint(8, 24), n_lo=n_lo, n_hi=_log_int(rng, 1e5, 1e6),
                nbins=rng.choice((512, 1024)), turns_lo=50, turns_hi=_log_int(rng, 150, 500), per_tick=rng.choice((50, 100)),
                sizes=rng.randrange(1000))


# -- what a case asks for ----------------------------------------------------

def _lattice(m, turns):
    """The parameters of a case or of a member; a pair's two voltages keep the phase of their mean."""
    on = m["flags"].split(",")
    flags = tuple(f in on for f in ("wake", "eta", "E0", "SR", "QE"))
    if m["lattice"] == "reference":
        return W.reference_benchmark_lattice(turns, flags)
    p = W.ring_3gev_lattice(turns, **({"voltage": m["V"]} if "V" in m else {}), flags=flags)
    p["voltage"] *= m.get("V_times", 1.0)
    return p


def _sigmas(case):
    return W.reference_benchmark_bunch_sigmas() if case["lattice"] == "reference" else (W.SIGMA_Z, W.SIGMA_E)


def _resonators(case):
    return [W.RESONATOR_BB, W.RESONATOR_LOWQ][:case["resonators"]]


def _members(case):
    """The bunches of a batch, or the jobs of a served mix (pairs as two): sizes and settings of each."""
    r = random.Random(case["sizes"])
    out = []
    while len(out) < case["count"]:
        n, V = _log_int(r, case["n_lo"], case["n_hi"]), r.uniform(2.5e6, 4.0e6)
        turns = case["turns"] if case["kind"] == "batch" else _log_int(r, case["turns_lo"], case["turns_hi"])
        q = _charge(r, turns)
        m = dict(n=n, turns=turns, V=V, nbins=case["nbins"], lattice="ring3", charge_nC=q, resonators=1, half_width=8.0,
                 flags=ALL_ON, monitor=False, stream=len(out), pair=0)
        if case["kind"] == "serve" and len(out) + 1 < case["count"] and r.random() < 0.1:
            out += [dict(m, V_times=1 - 0.005, pair=1), dict(m, V_times=1 + 0.005, pair=2)]
        else:
            out.append(m)
    return out


def _noise_seed(seed, stream=0):
    return (int(seed) * 1000003 + 7919 * stream + 1) % (1 << 62)


def _options(m, seed):
    return H.TrackingOptions(seed=_noise_seed(seed, m.get("stream", 0)), resonators=_resonators(m),
                             charge=m["charge_nC"] * 1e-9, bin_half_width_sigmas=m["half_width"], monitor=m["monitor"])


def _params(m):
    return H.SimulationParameters.from_dict(_lattice(m, m["turns"]))


def _gaussian(m, seed):
    """The bunch before the call, on the GPU."""
    g = torch.Generator(device="cuda")
    g.manual_seed(_noise_seed(seed, m.get("stream", 0)) % (1 << 40))
    sz, sE = _sigmas(m)
    z = torch.randn(m["n"], generator=g, device="cuda", dtype=torch.float64).mul_(sz)
    e = torch.randn(m["n"], generator=g, device="cuda", dtype=torch.float64).mul_(sE)
    return z, e


class _View:
    """One of a resident bunch's device arrays for torch; keeps the bunch."""

    def __init__(self, bunch, address):
        self.bunch = bunch
        self.__cuda_array_interface__ = {"shape": (bunch.n,), "typestr": "<f8", "data": (address, False), "version": 2}


def _bunch(m, seed):
    import ctypes
    from haissinskijulia_amd import _lib
    b = H.DeviceBunch(m["n"])
    zp, ep = ctypes.c_void_p(), ctypes.c_void_p()
    _lib.check(_lib.load().hm_bunch_device_ptrs(b._h, ctypes.byref(zp), ctypes.byref(ep)))
    z, e = (torch.as_tensor(_View(b, p.value), device="cuda") for p in (zp, ep))
    for to, x in zip((z, e), _gaussian(m, seed)):
        to.copy_(x)
    return b, z, e


def prepare(case, seed):
    s = {"kind": case["kind"]}
    if case["kind"] == "host":
        s["particles"] = H.Particles(*(x.cpu().numpy() for x in _gaussian(case, seed)))
        s["buffers"] = H.create_simulation_buffers(case["n"], case["nbins"])
        s["device"] = H.MI355X.default()
        s["params"], s["options"] = _params(case), _options(case, seed)
    elif case["kind"] == "resident":
        s["bunch"], s["z"], s["dE"] = _bunch(case, seed)
        s["nbins"], s["params"], s["options"] = case["nbins"], _params(case), _options(case, seed)
    elif case["kind"] == "batch":
        members = _members(case)
        s["bunches"], s["z"], s["dE"] = zip(*(_bunch(m, seed) for m in members))
        s["nbins"] = [m["nbins"] for m in members]
        s["params"], s["options"] = [_params(m) for m in members], [_options(m, seed) for m in members]
    else:
        s["server"] = H.Server(budget_bytes=200 << 30, max_slots=64)
        s["per_tick"] = case["per_tick"]
        s["jobs"] = []
        for m in _members(case):
            if m["pair"] == 2:
                continue   # submitted with its partner
            job = H.Job(params=_params(dict(m, V_times=1.0)), n=m["n"], nbins=m["nbins"],
                        particle_seed=_noise_seed(seed, 500 + m["stream"]), sigma_z=W.SIGMA_Z, sigma_E=W.SIGMA_E,
                        options=_options(m, seed))
            s["jobs"].append((job, m["pair"] == 1))
    torch.cuda.synchronize()
    return s


def _spreads(rs):
    return {k: np.array([getattr(r, k) for r in rs]) for k in ("sigma_E", "sigma_z", "E0")}


def run(s):
    if s["kind"] == "host":
        sE, sz, E0 = H.longitudinal_evolve(s["particles"], s["params"], s["buffers"], s["device"], True, s["options"])
        s["options"].turn_offset += s["params"].n_turns
        c = s["particles"].coordinates
        return {"z": c.z, "dE": c.dE, "sigma_E": sE, "sigma_z": sz, "E0": E0}
    if s["kind"] == "resident":
        r = s["bunch"].evolve(s["params"], s["nbins"], s["options"])
        s["options"].turn_offset += s["params"].n_turns
        out = {"z": s["z"], "dE": s["dE"], "sigma_E": r.sigma_E, "sigma_z": r.sigma_z, "E0": r.E0}
        if r.monitor is not None:
            out.update(zip(("turn_z", "turn_sigma_z", "turn_E0", "turn_count"), r.monitor.T))
        return out
    if s["kind"] == "batch":
        rs = H.batch_evolve(s["bunches"], s["nbins"], s["params"], s["options"])
        for o, p in zip(s["options"], s["params"]):
            o.turn_offset += p.n_turns
        return {"z": list(s["z"]), "dE": list(s["dE"]), **_spreads(rs)}
    ids = []
    for job, pair in s["jobs"]:
        ids += s["server"].submit_voltage_pair(job) if pair else (s["server"].submit(job),)
    done = {r.job_id: r for r in s["server"].run(s["per_tick"])}
    rs = [done[i] for i in ids]
    return {**_spreads([r.result for r in rs]), "centroid_z": np.array([r.centroid_z for r in rs]),
            "centroid_E": np.array([r.centroid_E for r in rs])}


def work(case):
    """Each turn reads and writes every particle's (z, dE) once: the next turn needs the whole bunch's line density.
    FP64 operations per particle and turn, elementary functions as their shortest usual polynomials: the RF kick 22,
    the drift 10 (16 with its own slippage), damping 1, excitation 32, line density 5, kick 9, E0 update 3."""
    members = _members(case) if case["kind"] in ("batch", "serve") else [case]
    nbytes = flops = 0.0
    for m in members:
        on = m["flags"].split(",")
        per = 22 + (16 if "eta" in on else 10) + ("SR" in on) + 32 * ("QE" in on) + 14 * ("wake" in on) + 3 * ("E0" in on)
        nbytes += 32.0 * m["n"] * m["turns"]
        flops += float(per) * m["n"] * m["turns"]
    return {"bytes": nbytes, "flops": flops}


# -- the same in plain torch -------------------------------------------------

def _philox(index, c2, stream, seed):
    """Philox4x32-10 (Salmon et al., SC'11) of the counters (index, c2, stream): four words per index."""
    low = 0xFFFFFFFF
    c = [index & low, index >> 32, torch.full_like(index, c2 & low), torch.full_like(index, stream)]
    k0, k1 = seed & low, (seed >> 32) & low
    for _ in range(10):
        p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
        c = [((p1 >> 32) & low) ^ c[1] ^ k0, p1 & low, ((p0 >> 32) & low) ^ c[3] ^ k1, p0 & low]
        k0, k1 = (k0 + 0x9E3779B9) & low, (k1 + 0xBB67AE85) & low
    return c


def _normals(index, c2, stream, seed):
    """Two normals per index (Box and Muller) from 53-bit uniforms."""
    x = _philox(index, c2, stream, seed)
    u1 = ((x[0] >> 5).double() * 67108864.0 + (x[1] >> 6).double() + 1.0) * 2.0 ** -53
    u2 = ((x[2] >> 5).double() * 67108864.0 + (x[3] >> 6).double()) * 2.0 ** -53
    r = torch.sqrt(-2.0 * torch.log(u1))
    return r * torch.cos(TWO_PI * u2), r * torch.sin(TWO_PI * u2)


def _std(x):
    n = x.numel()
    s, s2 = float(x.sum()), float((x * x).sum())
    return math.sqrt(max(0.0, (s2 / n - (s / n) ** 2) * n / (n - 1)))


def _resonator(s, Rs, fr, Q):
    """Chao, Physics of Collective Beam Instabilities, eq. 2.84 (Q > 1/2), half its jump at s = 0."""
    wr = TWO_PI * fr
    a = wr / (2 * Q)
    wb = math.sqrt(wr * wr - a * a)
    w = 2 * a * Rs * np.exp(-a * s / C_LIGHT) * (np.cos(wb * s / C_LIGHT) - (a / wb) * np.sin(wb * s / C_LIGHT))
    return np.where(s == 0, a * Rs, w)


def _track(m, z, e, noise_seed):
    p = _lattice(m, m["turns"])
    n, nb = z.numel(), m["nbins"]
    E0, mass, phis, h = p["E0"], p["mass"], p["phi_s"], p["harmonic"]
    sE0, sz0 = _std(e), _std(z)
    pairs = torch.arange((n + 1) // 2, device=z.device, dtype=torch.int64)
    wake, by_lag, q = p["use_wakefield"], m["resonators"] > 0, m["charge_nC"] * 1e-9
    if wake:
        zw = m["half_width"] * sz0
        step = 2 * zw / nb
        centres = (np.longdouble(zw) * (2 * np.arange(nb) + 1 - nb) / nb).astype(np.float64)
        c0, c1 = float(centres[0]), float(centres[-1])
        inv = 1.0 / ((c1 - c0) / (nb - 1))
        if by_lag:
            W_tab = sum(_resonator(np.arange(nb) * step, *r) for r in _resonators(m))
        else:
            b = p["pipe_radius"]
            wf, ws = ((120 * math.pi) * C_LIGHT) / (math.pi * b), math.sqrt(60.0 / b)
            W_tab = np.where(centres > 0, 0.0, wf * np.exp(np.minimum(centres, 0) / 4e-3) * np.cos(ws * centres))
        lam = np.ones(nb) if q > 0 else (1 / (math.sqrt(TWO_PI) * 0.15)) * np.exp(centres ** 2 * (-0.5 / 0.15 ** 2))
        lam = torch.from_numpy(lam).to(z.device)
        L = H.next_power_of_two(2 * nb)
        W_hat = torch.fft.rfft(torch.from_numpy(W_tab).to(z.device), n=L)
    seen = np.zeros((m["turns"], 4))
    for t in range(m["turns"]):
        g0 = E0 / mass
        b0 = math.sqrt(1.0 - 1.0 / (g0 * g0))
        rf = p["freq_rf"] * TWO_PI / (b0 * C_LIGHT)
        per_phase = TWO_PI * h / (b0 * b0 * E0)
        lost = 4 * 8.85e-5 * (E0 / 1e9) ** 3 / p["radius"]
        before = e
        e = e + p["voltage"] * (torch.sin(phis - z * rf) - math.sin(phis))
        if p["use_excitation"]:
            a, b = _normals(pairs, t, 0, noise_seed)
            e = e + math.sqrt(1 - (1 - lost) ** 2) * sE0 * torch.stack((a, b), 1).reshape(-1)[:n]
            del a, b
        if p["SR_damping"]:
            e = e * (1 - lost)
        if p["update_eta"]:
            eta = p["alpha_c"] - (g0 + e / mass) ** -2
        else:
            eta = p["alpha_c"] - 1.0 / (g0 * g0)
        phi = phis - z * rf + per_phase * eta * e
        z = (phis - phi) / rf
        del phi, eta
        if wake:
            mean = float(z.sum()) / n
            sz = _std(z)
            inside = (z >= -zw) & (z <= zw)
            counts = torch.bincount(((z[inside] + zw) * (1.0 / step)).long().clamp_(max=nb - 1), minlength=nb)
            n_h = int(counts.sum())
            if q > 0:
                current = q
            else:
                decade = 10.0 ** min(10, math.floor(math.log10(n)))
                current = (1e11 / decade) * n / E0 / (TWO_PI * p["radius"]) * sz / ((p["alpha_c"] - 1.0 / (g0 * g0)) * sE0 * sE0)
            g = lam * (counts.double() / n_h)
            if by_lag:   # a bin feels the bins ahead of it
                P = torch.fft.irfft(torch.fft.rfft(g.flip(0), n=L) * W_hat, n=L)[:nb].flip(0) * current
            else:
                P = torch.fft.irfft(torch.fft.rfft(g, n=L) * W_hat, n=L)[:nb] * current
            u = (z.clamp(c0, c1) - c0) * inv
            k = u.long().clamp_(max=nb - 2)
            u -= k
            e = e - (P[k] * (1.0 - u) + P[k + 1] * u)
            seen[t, 0], seen[t, 1], seen[t, 3] = mean, sz, n_h
            del u, k, inside
        if p["update_E0"]:
            change = float((e - before).sum()) / n
            E0 += change
            e = e - change
        seen[t, 2] = E0
    return z, e, E0, seen


def _exact_one(m, z, e, noise_seed):
    z, e, E0, seen = _track(m, z, e, noise_seed)
    out = {"z": z, "dE": e, "sigma_E": _std(e), "sigma_z": _std(z), "E0": E0}
    if m["monitor"]:
        out.update(zip(("turn_z", "turn_sigma_z", "turn_E0", "turn_count"), seen.T))
    return out


def exact(case, seed):
    """The same tracking in plain torch; None where its turns would take too long."""
    if case["kind"] in ("host", "resident"):
        z, e = _gaussian(case, seed)
        out = _exact_one(case, z, e, _noise_seed(seed))
        return {k: v.cpu().numpy() for k, v in out.items() if k in ("z", "dE")} | {
            k: v for k, v in out.items() if k not in ("z", "dE")} if case["kind"] == "host" else out
    members = _members(case)
    if sum(m["turns"] * (1.0 + m["n"] / 2e6) for m in members) > 12000:
        return None
    outs = []
    for m in members:
        if case["kind"] == "batch":
            z, e = _gaussian(m, seed)
            outs.append(_exact_one(m, z, e, _noise_seed(seed, m["stream"])))
        else:   # a served job's bunch: two normals of the stream of its particle seed per particle
            i = torch.arange(m["n"], device="cuda", dtype=torch.int64)
            a, b = _normals(i, 0, 1, _noise_seed(seed, 500 + m["stream"]))
            o = _exact_one(m, W.SIGMA_Z * a, W.SIGMA_E * b, _noise_seed(seed, m["stream"]))
            outs.append(dict({k: o[k] for k in ("sigma_E", "sigma_z", "E0")},
                             centroid_z=float(o["z"].mean()), centroid_E=float(o["dE"].mean())))
    spread = {k: np.array([o[k] for o in outs]) for k in ("sigma_E", "sigma_z", "E0")}
    if case["kind"] == "batch":
        return {"z": [o["z"] for o in outs], "dE": [o["dE"] for o in outs], **spread}
    return {**spread, "centroid_z": np.array([o["centroid_z"] for o in outs]),
            "centroid_E": np.array([o["centroid_E"] for o in outs])}
