"""The potential at the centre of a Hernquist subhalo (its gradient has no value there) and where
r^2 overflows: - G m / a and 0 beside the host's and the other subhalos' parts, in the launch shapes
for few and many points and whatever else is asked for."""
import numpy as np
import pytest
import torch

from test_gpu_core import bound_orbits

pytestmark = pytest.mark.gpu

G = 4.498502151469553e-12


@pytest.mark.parametrize("n", [5, 200_000])
def test_hernquist_centre(ssc, n):
    from streamsculptor_amd import workloads as W
    from streamsculptor_amd.main import usys
    from streamsculptor_amd.potential import (HernquistPotential, Potential_Combine,
                                              SubhaloLinePotentialCustom_fromFunc)
    rng = np.random.default_rng(n)
    m = 6
    mass, rs = 10 ** rng.uniform(6, 8, m), rng.uniform(0.1, 1.0, m)
    x0, v = rng.normal(scale=10.0, size=(m, 3)), rng.normal(scale=0.2, size=(m, 3))
    host = W.host_potential()
    sub = SubhaloLinePotentialCustom_fromFunc(HernquistPotential, mass, rs, x0, v, np.zeros(m),
                                              np.full(m, 100.0), units=usys)
    pot = Potential_Combine([host, sub], units=usys)
    x = bound_orbits(rng, n)[:, :3]
    x[:m - 1] = x0[:min(n, m - 1)]
    print(f"[eval] Hernquist centres among {n} points", flush=True)
    r = np.linalg.norm(x[:, None] - x0, axis=2)
    ref = host.potential(x, 0.0).cpu().numpy() - (G * mass / (r + rs)).sum(1)
    assert (r.min(1)[:m - 1] == 0.0).all()
    phi = pot.potential(x, 0.0).cpu().numpy()
    np.testing.assert_allclose(phi, ref, rtol=1e-13)


def test_far_away(ssc):
    from streamsculptor_amd import workloads as W  # noqa: F401
    from streamsculptor_amd.main import usys
    from streamsculptor_amd.potential import (HernquistPotential, PlummerPotential,
                                              Potential_Combine,
                                              SubhaloLinePotentialCustom_fromFunc)
    sub = SubhaloLinePotentialCustom_fromFunc(HernquistPotential, np.array([1e8]), np.array([0.5]),
                                              np.zeros((1, 3)), np.zeros((1, 3)), np.zeros(1),
                                              np.full(1, 100.0), units=usys)
    host = PlummerPotential(m=1e10, r_s=2.0, units=usys)
    x = np.array([[1e200, 0.0, 0.0]])
    print("[eval] r^2 beyond the largest number", flush=True)
    assert torch.equal(Potential_Combine([host, sub], units=usys).potential(x, 0.0),
                       host.potential(x, 0.0))
