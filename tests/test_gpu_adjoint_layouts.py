"""The discrete adjoint with sources over its launch shapes: lane groups of 8, 16 and 32 in the
source adjoints (the largest table of each, one past it, several passes over the table), chunks
of particles that end inside a tile, one particle, particles that never move, and the lanes per
orbit with and without start rows.  lam0 and the gradients with respect to the host parameters,
the source masses and the source positions against the oracle, <= 1e-9 relative."""
import numpy as np
import pytest
import torch

from test_gpu_core import bound_orbits

pytestmark = pytest.mark.gpu

G = 4.498502151469553e-12


def _rel(a, b):
    a = a.cpu().numpy() if isinstance(a, torch.Tensor) else np.asarray(a)
    return np.linalg.norm(a.reshape(-1) - b.reshape(-1)) / max(np.linalg.norm(b), 1e-300)


@pytest.mark.parametrize("kind,m,n,nsteps,every,ragged", [
    ("track", 1, 1, 7, 3, False),
    ("track", 16, 65, 23, 10, True),     # 8 lanes a group, two sources each: the largest table
    ("track", 17, 130, 23, 10, False),   # 16 lanes
    ("static", 32, 700, 21, 10, True),
    ("static", 33, 13000, 8, 4, True),   # 32 lanes; 128 particles a chunk, the last one short
    ("static", 64, 300, 25, 10, False),
    ("track", 65, 3000, 12, 5, True),    # two passes; chunks no shorter than the table
    ("static", 200, 1000, 12, 12, True),
    ("track", 67, 4097, 9, 1, False),    # every row stored; 8 lanes an orbit
])
def test_adjoint_shapes(oracle, ssc, kind, m, n, nsteps, every, ragged):
    from streamsculptor_amd import _lib
    from streamsculptor_amd import workloads as W
    from streamsculptor_amd.adjoint import LeapfrogAdjoint
    from streamsculptor_amd.main import SourceSet
    rng = np.random.default_rng(1000 + n + m)
    host, h = W.host_potential(), oracle.host(W.host_components())
    gm, rs = G * 10 ** rng.uniform(6.0, 7.5, m), rng.uniform(0.1, 0.6, m)
    t0, dt = -float(nsteps), 1.0
    if kind == "static":
        pos = rng.normal(scale=10.0, size=(m, 3))
        src = SourceSet(_lib.SRC_STATIC, gm=gm, rs=rs, pos=pos)
        so = oracle.Sources(oracle.SRC_STATIC, gm=gm, rs=rs, pos=pos)
    else:
        pos = (rng.normal(scale=10.0, size=(1, m, 3))
               + 0.1 * np.arange(nsteps + 1)[:, None, None] * rng.normal(size=(1, m, 3)))
        src = SourceSet(_lib.SRC_TRACK, gm=gm, rs=rs, pos=pos, grid=(t0, dt))
        so = oracle.Sources(oracle.SRC_TRACK, gm=gm, rs=rs, pos=pos)
    w0 = bound_orbits(rng, n)
    start = np.sort(rng.integers(0, nsteps + 3, n)).astype(np.int32) if ragged else None
    lam = rng.normal(size=(n, 6))
    print(f"[adjoint layouts] {kind} m={m} n={n}", flush=True)
    adj = LeapfrogAdjoint(host, w0, t0, dt, nsteps, start=start, checkpoint_every=every, src=src)
    wT = adj.forward()
    out = adj.backward(lam)
    torch.cuda.synchronize()
    ref = oracle.adjoint_leapfrog(h, w0, t0, dt, nsteps, lam, start=start, src=so)
    fwd = oracle.leapfrog(h, w0, t0, dt, nsteps, start=start, src=so)
    assert _rel(wT, fwd) <= 1e-9
    e = {k: _rel(out[k], ref[k]) for k in ("lam0", "g_host", "g_gm", "g_pos")}
    assert all(v <= 1e-9 for v in e.values()), e
