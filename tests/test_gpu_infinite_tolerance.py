"""Adaptive steps without error control: an infinite absolute tolerance, whose error scale is
infinite, takes every step that dtmax allows, as a tolerance does that no error reaches (1e290: all
scaled errors underflow) -- the same rows bit for bit, for orbits and for responses."""
import numpy as np
import pytest
import torch

from test_gpu_core import bound_orbits

pytestmark = pytest.mark.gpu

G = 4.498502151469553e-12


@pytest.mark.parametrize("rtol", [0.0, 1e-7])
def test_orbits(ssc, rtol):
    from streamsculptor_amd import workloads as W
    from streamsculptor_amd.adaptive import dopri5
    host = W.host_potential()
    w0 = bound_orbits(np.random.default_rng(3), 70)
    ts = np.linspace(0.0, 300.0, 7)
    print(f"[infinite tolerance] orbits, rtol {rtol}", flush=True)
    a, b = (dopri5(host, w0, 0.0, 300.0, ts=ts, rtol=rtol, atol=atol, dtmin=None, dtmax=2.0,
                   max_steps=400, throw=False) for atol in (float("inf"), 1e290))
    for x, y in zip(a, b):
        if torch.is_tensor(x):
            assert torch.isfinite(x.double()).all() and torch.equal(x, y)


@pytest.mark.parametrize("m", [5, 40])  # groups of one wave and of two
def test_responses(ssc, m):
    from streamsculptor_amd import _lib
    from streamsculptor_amd import workloads as W
    from streamsculptor_amd.fields import perturb_dopri5
    from streamsculptor_amd.main import SourceSet
    rng = np.random.default_rng(m)
    gm = G * 10 ** rng.uniform(6, 8, m)
    src = SourceSet(_lib.SRC_STATIC, gm=gm, rs=1.62 * np.sqrt(gm / G / 1e8),
                    pos=rng.normal(scale=10.0, size=(m, 3)))
    w0 = bound_orbits(rng, 9)
    print(f"[infinite tolerance] responses to {m} subhalos", flush=True)
    a, b = (perturb_dopri5(W.host_potential(), src, w0, None, 100.0, with_radius=True, rtol=1e-7,
                           atol=atol, dtmin=0.0, dtmax=2.0, max_steps=200, throw=False)
            for atol in (float("inf"), 1e290))
    assert (a[4][:, 2] == 0).all()
    for x, y in ((a[0], b[0]), (a[1], b[1]), (a[4], b[4])):
        assert torch.isfinite(x.double()).all() and torch.equal(x, y)
