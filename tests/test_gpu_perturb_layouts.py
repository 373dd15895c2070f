"""Lane layouts of the adaptive response kernel: group widths at the edges of a wave and of the
block (narrow groups without barriers, groups of two and four waves), and hosts of more
components than a group has waves.  Kernel vs oracle on the same inputs, <= 1e-6 relative (the
adaptive bar), step counts equal."""
import numpy as np
import pytest

from test_gpu_core import bound_orbits
from test_gpu_perturb_dopri5 import G, _rel, _sources

pytestmark = pytest.mark.gpu


def _components(nc):
    from streamsculptor_amd import workloads as W
    extra = [(4, [G * 2e9, 2.0]), (3, [G * 1.7e9, 0.07, 0.0]), (1, [G * 5e9, 4.0, 0.4]),
             (2, [G * 1e10, 9.0]), (4, [G * 1e9, 30.0])]
    return (W.host_components() + extra)[:nc] if nc > 1 else [(2, [G * 5.4e11, 15.62])]


def _potential(comps):
    from streamsculptor_amd.main import Potential

    class Host(Potential):
        def __init__(self):
            super().__init__(None, {})

        def _kernel_components(self):
            return [(k, list(p)) for k, p in comps]

    return Host()


@pytest.mark.parametrize("kind,radius,m,n,nc", [
    ("line", False, 1, 70, 3),         # 8 lanes, blocks of 32 particles, the last one partial
    ("line", False, 9, 33, 8),         # 16 lanes
    ("hernquist", True, 16, 17, 1),    # 32 lanes, one host component
    ("line", False, 64, 9, 5),         # 64 lanes: the widest group without barriers
    ("line", True, 33, 5, 3),          # 66 vectors: two waves, three components
    ("hernquist", False, 128, 3, 8),   # two waves, eight components: four each
    ("static", True, 65, 2, 8),        # 130 vectors: four waves, two components each
    ("line", False, 256, 1, 2),        # the block full, waves without a component
])
def test_layouts_match_oracle(oracle, ssc, kind, radius, m, n, nc):
    from streamsculptor_amd.fields import perturb_dopri5
    rng = np.random.default_rng(100 + m)
    comps = _components(nc)
    src, so = _sources(oracle, kind, rng, m, 0.0, 400.0)
    w0 = bound_orbits(rng, n)
    dw0 = rng.normal(scale=1e-3, size=(n, m, 12 if radius else 6))
    t_start = np.sort(rng.uniform(0.0, 200.0, n))
    tol = dict(rtol=1e-7, atol=1e-7, dtmin=0.05, max_steps=20_000)
    print(f"[layouts] {kind} radius={radius} m={m} n={n} components={nc}", flush=True)
    w, dw, _, _, st = perturb_dopri5(_potential(comps), src, w0, dw0, 400.0, t_start=t_start,
                                     with_radius=radius, **tol)
    wr, dwr, _, _, sto = oracle.perturb_dopri5(oracle.host(comps), so, w0, 400.0,
                                               t_start=t_start, dw0=dw0, with_radius=radius, **tol)
    assert (sto[:, 2] == 0).all()
    assert _rel(w, wr) <= 1e-6 and _rel(dw, dwr) <= 1e-6
    assert (st.cpu().numpy() == sto).all(axis=1).mean() >= 0.97
