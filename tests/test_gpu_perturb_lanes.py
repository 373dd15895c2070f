"""The split response kernel over its launch shapes: two, four or eight responses per lane (the
rule on particles and sources), the largest source counts of each, particles that do not fill a
wave or a block, and workspaces of one row (one buffer), two and three rows (two buffers of one
row) and all rows.  Final rows and responses against the oracle on a sample of the particles,
<= 1e-9 relative; other workspaces bit for bit."""
import numpy as np
import pytest
import torch

from test_gpu_core import bound_orbits

pytestmark = pytest.mark.gpu

G = 4.498502151469553e-12


def _rel(a, b):
    a, b = a.reshape(len(a), -1), b.reshape(len(b), -1)
    return (np.linalg.norm(a - b, axis=1) / np.maximum(np.linalg.norm(b, axis=1), 1e-300)).max()


@pytest.mark.parametrize("kind,radius,m,n,nsteps", [
    ("static", False, 1, 3, 40),        # two per lane, one source
    ("static", False, 5, 65, 30),       # a wave and one particle, lanes without a response
    ("line", False, 512, 7, 12),        # two per lane at 256 lanes
    ("line", False, 513, 7, 12),        # eight per lane
    ("static", True, 512, 5, 12),       # two per lane with the radius block
    ("static", True, 513, 5, 12),       # four
    ("hernquist", True, 1024, 3, 8),    # four per lane at 256 lanes
    ("static", False, 8, 131071, 5),    # the last size with two per lane ...
    ("static", False, 8, 131072, 5),    # ... and the first with eight
    ("line", False, 64, 16411, 5),      # eight, a partial last block
])
def test_split_shapes(oracle, ssc, kind, radius, m, n, nsteps):
    from streamsculptor_amd import _lib
    from streamsculptor_amd import workloads as W
    from streamsculptor_amd.fields import perturb_leapfrog
    from streamsculptor_amd.main import SourceSet
    rng = np.random.default_rng(n + m)
    host, h = W.host_potential(), oracle.host(W.host_components())
    gm = G * 10 ** rng.uniform(6, 8, m)
    kw = dict(gm=gm, rs=1.62 * np.sqrt(gm / G / 1e8), pos=rng.normal(scale=10.0, size=(m, 3)))
    kk, ko = {"static": (_lib.SRC_STATIC, oracle.SRC_STATIC),
              "line": (_lib.SRC_LINE, oracle.SRC_LINE),
              "hernquist": (_lib.SRC_LINE_HERNQUIST, oracle.SRC_LINE_HERNQUIST)}[kind]
    if kind != "static":
        kw.update(vel=rng.normal(scale=0.2, size=(m, 3)), t0=rng.uniform(0, nsteps, m),
                  t_window=rng.uniform(2, nsteps, m))
    src, so = SourceSet(kk, **kw), oracle.Sources(ko, **kw)
    w0 = bound_orbits(rng, n)
    dw0 = rng.normal(scale=1e-3, size=(n, m, 12 if radius else 6))
    start = np.sort(rng.integers(0, nsteps + 2, n)).astype(np.int32)
    print(f"[split] {kind} radius={radius} m={m} n={n}", flush=True)
    w, dw = perturb_leapfrog(host, src, w0, dw0, start, 0.0, 1.0, nsteps, radius)
    sel = np.unique(np.concatenate([[0, n - 1], rng.integers(0, n, 60)]))
    wr, dwr = oracle.perturb_leapfrog(h, so, w0[sel], 0.0, 1.0, nsteps, dw0=dw0[sel],
                                      start=start[sel], with_radius=radius)
    at = torch.as_tensor(sel, device=w.device)
    assert _rel(w[at].cpu().numpy(), wr) <= 1e-9
    assert _rel(dw[at].cpu().numpy(), dwr) <= 1e-9
    for rows in (1, 2, 3, nsteps + 1):
        w2, dw2 = perturb_leapfrog(host, src, w0, dw0, start, 0.0, 1.0, nsteps, radius,
                                   segment_rows=rows)
        assert torch.equal(w2, w) and torch.equal(dw2, dw), rows
