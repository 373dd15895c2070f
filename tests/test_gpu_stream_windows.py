"""Windowed streams: releases in potentials whose sources depend on the release time (a TRACK
table's rows, straight lines' positions), taken window by window from what is formed once for the
whole stream, and the memory of a window's new particles, which is read on another stream than the
one that wrote it."""
import numpy as np
import pytest
import torch

from test_gpu_core import bound_orbits

pytestmark = pytest.mark.gpu

G = 4.498502151469553e-12


def _potentials(t0, steps):
    """The host, and the host with live subhalos (TRACK) and with straight-line subhalos (LINE,
    some outside their windows at any time)."""
    from streamsculptor_amd import workloads as W
    from streamsculptor_amd.main import usys
    from streamsculptor_amd.potential import (LiveSubhaloPotential, Potential_Combine,
                                              SubhaloLinePotential)
    host = W.host_potential()
    live = LiveSubhaloPotential.from_orbits(host, *W.subhalo_ics(n=16, seed=2), t0, 1.0, steps)
    rng = np.random.default_rng(5)
    line = SubhaloLinePotential(10 ** rng.uniform(6, 8, 24), rng.uniform(0.1, 0.5, 24),
                                rng.normal(scale=15.0, size=(24, 3)),
                                rng.normal(scale=0.2, size=(24, 3)), rng.uniform(t0, 0, 24),
                                rng.uniform(50, 200, 24), units=usys)
    return host, {k: Potential_Combine([host, p], units=usys)
                  for k, p in (("track", live), ("line", line))}


@pytest.mark.parametrize("kind", ["track", "line"])
def test_releases_by_window(ssc, kind):
    """Progenitor and particles in the host alone, so that windows and one pass take the same
    steps: rows equal bit for bit, for two particles a step and for many."""
    from streamsculptor_amd import workloads as W
    from streamsculptor_amd.streams import gen_stream, spray_particles, spray_stream
    ts = np.linspace(-400.0, 0.0, 401)
    host, pots = _potentials(float(ts[0]), 400)
    rel = pots[kind]
    back = host.integrate_orbit(w0=W.PROG_TODAY, ts=[0.0, ts[0]], t0=0.0, t1=float(ts[0]),
                                solver="leapfrog", dt0=1.0).ys[-1]
    msat = np.linspace(2e5, 2e4, ts.size)
    print(f"[windows] releases among {kind} subhalos", flush=True)
    w0, start, _, (t0, dt, nsteps, _) = spray_particles(host, rel, ts, back, msat, 3, 7, 1.0)
    plain, *_ = spray_particles(host, host, ts, back, msat, 3, 7, 1.0)
    assert not torch.equal(w0, plain)  # the subhalos do enter the release
    one, _ = host._leapfrog(w0, t0, dt, nsteps, start=start)
    for chunks in (3, 8):
        assert torch.equal(spray_stream(host, rel, ts, back, msat, 3, 7, 1.0, chunks=chunks), one)
    if kind == "track":  # one pass for LINE: not static in time
        a = gen_stream(host, rel, ts, back, msat, 3, solver="leapfrog", dt0=1.0, chunks=5)
        b = gen_stream(host, rel, ts, back, msat, 3, solver="leapfrog", dt0=1.0, chunks=1)
        assert all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("kind", ["track", "line"])
def test_release_lanes(oracle, ssc, kind):
    """16 lanes a release over TRACK rows and LINE windows, against the oracle (<= 1e-11, as for
    static sources)."""
    from streamsculptor_amd import workloads as W
    rng = np.random.default_rng(8)
    host, pots = _potentials(-400.0, 400)
    pot = pots[kind]
    h = oracle.host(W.host_components())
    n, nseed = 37, 3
    w, msat, t = bound_orbits(rng, n), np.full(n, 2e4), np.linspace(-400.0, -7.0, n).round()
    _, src = pot._descriptor()
    d = {k: v.cpu().numpy() for k, v in src.tensors().items() if v is not None}
    steps = None
    if kind == "track":
        osrc, steps = oracle.Sources(oracle.SRC_TRACK, **d), (t + 400.0).astype(np.int32)
    else:
        osrc = oracle.Sources(oracle.SRC_LINE, **d)
        on = np.abs(t[:, None] - d["t0"]) < d["t_window"]
        assert on.any() and not on.all()
    print(f"[windows] release lanes, {kind}", flush=True)
    dev = torch.device("cuda")
    rows = pot._release_seeds(torch.as_tensor(w, device=dev),
                              torch.arange(n, dtype=torch.int32, device=dev),
                              torch.as_tensor(G * msat, device=dev), 4, nseed, 1.0, t_rel=t)
    rows = rows.cpu().numpy()
    for s in range(nseed):
        pc, pf, vc, vf = oracle.release(h, w, t, msat, 4 + s, src=osrc, steps=steps)
        for arm, (p, v) in enumerate(((pc, vc), (pf, vf))):
            ref = np.hstack([p, v])
            assert (np.abs(rows[s, arm] - ref).max(0) / np.abs(ref).max(0)).max() <= 1e-11


def test_new_particles_are_kept_while_read(ssc):
    """The first window's new particles are handed to ``integrate`` as they are; the second stream
    is kept busy after reading starts, and meanwhile nothing allocated on the third stream may get
    their memory."""
    from streamsculptor_amd import workloads as W
    from streamsculptor_amd.streams import _side_stream, spray_stream
    ts = np.linspace(-64.0, 0.0, 65)
    host = W.host_potential()
    back = host.integrate_orbit(w0=W.PROG_TODAY, ts=[0.0, ts[0]], t0=0.0, t1=float(ts[0]),
                                solver="leapfrog", dt0=1.0).ys[-1]
    first = []

    def integrate(w, t_start, step, n, start):
        if not first:
            first.append((w.data_ptr(), w.numel() * 8))
            torch.cuda._sleep(200_000_000)  # about a tenth of a second
        return host._leapfrog(w, t_start, step, n, start=start)[0]

    print("[windows] memory of new particles", flush=True)
    out = spray_stream(host, host, ts, back, W.MSAT, 1, 6, 1.0, integrate=integrate)
    done = torch.cuda.Event()
    done.record(_side_stream(out.device))
    lo, size = first[0]
    with torch.cuda.stream(_side_stream(out.device, 1)):
        got = [torch.empty(size // 8, dtype=torch.float64, device=out.device) for _ in range(64)]
    busy = not done.query()
    assert all(g.data_ptr() + size <= lo or g.data_ptr() >= lo + size for g in got)
    assert busy  # the second stream was still at work, so the assertion above was to the point
    torch.cuda.synchronize()
    assert torch.equal(out, spray_stream(host, host, ts, back, W.MSAT, 1, 6, 1.0))
