"""The response kernel's segments: grids of one segment, of two and of eight, and more room than
they want -- the same bits as with one row at a time, where nothing runs beside anything."""
import numpy as np
import pytest
import torch

from test_gpu_core import bound_orbits

pytestmark = pytest.mark.gpu

G = 4.498502151469553e-12


@pytest.mark.parametrize("n,nsteps", [(70, 127), (70, 128), (300, 600)])
def test_segments(ssc, n, nsteps):
    from streamsculptor_amd import _lib
    from streamsculptor_amd import workloads as W
    from streamsculptor_amd.fields import perturb_leapfrog
    from streamsculptor_amd.main import SourceSet
    rng = np.random.default_rng(nsteps)
    m = 9
    gm = G * 10 ** rng.uniform(6, 8, m)
    src = SourceSet(_lib.SRC_STATIC, gm=gm, rs=1.62 * np.sqrt(gm / G / 1e8),
                    pos=rng.normal(scale=10.0, size=(m, 3)))
    w0, start = bound_orbits(rng, n), np.sort(rng.integers(0, nsteps, n)).astype(np.int32)
    print(f"[segments] {n} particles, {nsteps} steps", flush=True)
    want = perturb_leapfrog(W.host_potential(), src, w0, None, start, 0.0, 1.0, nsteps, False,
                            segment_rows=1)
    for rows in (None, nsteps + 1):
        got = perturb_leapfrog(W.host_potential(), src, w0, None, start, 0.0, 1.0, nsteps, False,
                               segment_rows=rows)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
