"""The fixed-step stepper over its launch shapes with sources: one wave per orbit up to its last
size, every number of lanes per orbit (source counts that are no multiple of four times the
lanes, so that the blocks of four sources leave remainders), the sizes beside which the rule
changes, whole rounds of waves at one lane per orbit with the remainder at several, and two
orbits per lane for batches that fill the chip several times over.
Ragged starts, saved rows, and the same rows by the entry point for a stream's window, whose rule
the sizes are those of; against the oracle on a sample of the orbits, <= 1e-9 relative."""
import numpy as np
import pytest
import torch

from test_gpu_core import bound_orbits

pytestmark = pytest.mark.gpu

G = 4.498502151469553e-12


def _rel(a, b):
    return (np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)).max()


@pytest.mark.parametrize("kind,m,n,nsteps", [
    ("static", 64, 1024, 60),      # one wave per orbit, the last size ...
    ("static", 64, 1025, 60),      # ... and the first with 16 lanes an orbit
    ("static", 8, 1024, 60),       # the smallest table of the wave kernel ...
    ("line", 7, 1024, 60),         # ... and the largest of the lane groups
    ("tracked", 67, 4096, 40),     # 16 lanes, one wave per SIMD exactly, 67 = 16 x 4 + 3 sources
    ("tracked", 67, 4097, 40),     # 8 lanes
    ("static", 1, 1300, 40),       # one lane, one source
    ("line", 5, 300, 40),          # fewer sources than four per lane
    ("tracked", 13, 16384, 30),    # 4 lanes, one wave per SIMD exactly
    ("tracked", 13, 16385, 30),    # 2 lanes
    ("hernquist", 31, 32769, 20),  # one lane past two lanes' last size
    ("static", 515, 25000, 12),    # 4 lanes, two waves per SIMD
    ("static", 21, 393215, 4),     # the last size without pairs of orbits
    ("static", 21, 400000, 4),     # pairs would cost a round of waves
    ("static", 21, 524288, 4),     # two orbits per lane
    ("tracked", 64, 65537, 12),    # one lane each, and one orbit more with 16
    ("tracked", 13, 70001, 12),    # ... and a remainder that ends inside a block
    ("static", 100, 131500, 6),    # two whole rounds and a remainder
])
def test_launch_shapes(oracle, ssc, kind, m, n, nsteps):
    from streamsculptor_amd import _lib
    from streamsculptor_amd import workloads as W
    from streamsculptor_amd.main import SourceSet
    rng = np.random.default_rng(n + m)
    host, h = W.host_potential(), oracle.host(W.host_components())
    gm, rs = G * 10 ** rng.uniform(6.0, 7.5, m), rng.uniform(0.05, 0.6, m)
    t0, dt = -30.0, 1.0
    if kind == "static":
        pos = rng.normal(scale=10.0, size=(m, 3))
        src = SourceSet(_lib.SRC_STATIC, gm=gm, rs=rs, pos=pos)
        osrc = oracle.Sources(oracle.SRC_STATIC, gm=gm, rs=rs, pos=pos)
    elif kind == "tracked":
        pos = (rng.normal(scale=10.0, size=(1, m, 3))
               + 0.1 * np.arange(nsteps + 1)[:, None, None] * rng.normal(size=(1, m, 3)))
        src = SourceSet(_lib.SRC_TRACK, gm=gm, rs=rs, pos=pos, grid=(t0, dt))
        osrc = oracle.Sources(oracle.SRC_TRACK, gm=gm, rs=rs, pos=pos)
    else:
        pos, vel = rng.normal(scale=9.0, size=(m, 3)), rng.normal(scale=0.2, size=(m, 3))
        tc, tw = rng.uniform(t0, t0 + nsteps, m), rng.uniform(3, 30, m)
        sk, ok = ((_lib.SRC_LINE, oracle.SRC_LINE) if kind == "line"
                  else (_lib.SRC_LINE_HERNQUIST, oracle.SRC_LINE_HERNQUIST))
        src = SourceSet(sk, gm=gm, rs=rs, pos=pos, vel=vel, t0=tc, t_window=tw)
        osrc = oracle.Sources(ok, gm=gm, rs=rs, pos=pos, vel=vel, t0=tc, t_window=tw)
    w0 = bound_orbits(rng, n)
    start = np.sort(rng.integers(0, nsteps + 2, n)).astype(np.int32)
    start[0] = 0
    print(f"[leapfrog lanes] {kind} m={m} n={n}", flush=True)
    save = [0, nsteps // 2, nsteps]
    hd, _ = host._descriptor()
    sd = src.desc()
    wd, st = _lib.f64(w0), _lib.i32(start)
    si = _lib.i32(save)
    out = torch.empty_like(wd)
    ys = torch.empty(len(save), n, 6, dtype=torch.float64, device=wd.device)
    _lib.call("ssc_leapfrog", _lib.ctypes.byref(hd), _lib.ctypes.byref(sd), _lib.ptr(wd),
              _lib.ptr(st), n, t0, dt, nsteps, _lib.ptr(out), _lib.ptr(si), len(save),
              _lib.ptr(ys))
    # the same starts through the launch shaped for orbits that all walk the whole window
    win = torch.empty_like(wd)
    _lib.call("ssc_leapfrog_window", _lib.ctypes.byref(hd), _lib.ctypes.byref(sd), _lib.ptr(wd),
              _lib.ptr(st), n, t0, dt, nsteps, _lib.ptr(win))
    torch.cuda.synchronize()
    pick = np.unique(np.concatenate([[0, n - 1], rng.integers(0, n, 250)]))
    final, traj = oracle.leapfrog(h, w0[pick], t0, dt, nsteps, start=start[pick], src=osrc,
                                  traj=True)
    assert _rel(out.cpu().numpy()[pick], final) <= 1e-9
    assert _rel(win.cpu().numpy()[pick], final) <= 1e-9
    for k, y in zip(save, ys.cpu().numpy()):
        assert _rel(y[pick], traj[k]) <= 1e-9
