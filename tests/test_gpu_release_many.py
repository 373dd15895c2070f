"""One seed of many releases, a lane each (from 32,768 releases on): against the oracle, <= 1e-11
relative as the other launch shapes, and in the host alone bit for bit the rows of a launch one
release shorter, whose lanes share the work."""
import numpy as np
import pytest
import torch

from test_gpu_core import bound_orbits

pytestmark = pytest.mark.gpu

G = 4.498502151469553e-12


@pytest.mark.parametrize("kind,n", [("host", 32768), ("host", 33000), ("static", 32768),
                                    ("line", 32769)])
def test_many_releases(oracle, ssc, kind, n):
    from streamsculptor_amd import workloads as W
    from streamsculptor_amd.main import usys
    from streamsculptor_amd.potential import (HernquistPotential, PlummerClumps, Potential_Combine,
                                              SubhaloLinePotentialCustom_fromFunc)
    rng = np.random.default_rng(n)
    host, m = W.host_potential(), 9
    mass, rs = 10 ** rng.uniform(6.0, 7.5, m), rng.uniform(0.05, 0.6, m)
    pos = rng.normal(scale=12.0, size=(m, 3))
    t = np.linspace(-300.0, 0.0, n)
    pot, src = host, None
    if kind == "static":
        pot = Potential_Combine([host, PlummerClumps(mass, rs, pos, units=usys)], units=usys)
        src = oracle.Sources(oracle.SRC_STATIC, gm=G * mass, rs=rs, pos=pos)
    elif kind == "line":
        vel, tc, tw = rng.normal(scale=0.2, size=(m, 3)), rng.uniform(-300, 0, m), np.full(m, 60.0)
        pot = Potential_Combine([host, SubhaloLinePotentialCustom_fromFunc(
            HernquistPotential, mass, rs, pos, vel, tc, tw, units=usys)], units=usys)
        src = oracle.Sources(oracle.SRC_LINE_HERNQUIST, gm=G * mass, rs=rs, pos=pos, vel=vel, t0=tc,
                             t_window=tw)
    w, msat = bound_orbits(rng, n), np.full(n, 2e4)
    dev = torch.device("cuda")

    def release(k):
        return pot._release(torch.as_tensor(w[:k], device=dev),
                            torch.arange(k, dtype=torch.int32, device=dev),
                            torch.as_tensor(G * msat[:k], device=dev), 7, 1.0, t_rel=t[:k])

    print(f"[many releases] {kind} {n}", flush=True)
    got = release(n)
    for a, b in zip(got, oracle.release(oracle.host(W.host_components()), w, t, msat, 7, src=src)):
        assert (np.abs(a.cpu().numpy() - b).max(0) / np.abs(b).max(0)).max() <= 1e-11
    if kind == "host":
        assert all(torch.equal(a[:32767], b) for a, b in zip(got, release(32767)))
