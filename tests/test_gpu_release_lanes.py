"""The release kernel over its launch shapes: 1, 16 or 64 lanes a release by the size of the
source table, release counts around the blocks' 8 and 16, one seed, seeds that do not fill a
block's round and seeds shared by several blocks; against the oracle's release for a few of the
seeds, <= 1e-11 relative (the tidal radius is a cube root of a difference of two sums)."""
import numpy as np
import pytest
import torch

from test_gpu_core import bound_orbits

pytestmark = pytest.mark.gpu

G = 4.498502151469553e-12


@pytest.mark.parametrize("m,n,nseed", [
    (0, 1, 1), (0, 15, 5), (0, 17, 300), (1, 16, 3), (63, 33, 9),
    (64, 7, 1), (64, 8, 40), (130, 9, 600), (515, 1025, 2),
])
def test_release_shapes(oracle, ssc, m, n, nseed):
    from streamsculptor_amd import workloads as W
    from streamsculptor_amd.potential import PlummerClumps, Potential_Combine
    rng = np.random.default_rng(100 + m + n)
    pot, osrc = W.host_potential(), None
    h = oracle.host(W.host_components())
    if m:
        pos, mass = rng.normal(scale=12.0, size=(m, 3)), 10 ** rng.uniform(6.0, 7.5, m)
        rs = rng.uniform(0.05, 0.6, m)
        pot = Potential_Combine([pot, PlummerClumps(mass, rs, pos, units=ssc.usys)],
                                units=ssc.usys)
        osrc = oracle.Sources(oracle.SRC_STATIC, gm=G * mass, rs=rs, pos=pos)
    w = bound_orbits(rng, n)
    msat = np.full(n, 2e4)
    seed0 = 11
    print(f"[release lanes] m={m} n={n} nseed={nseed}", flush=True)
    dev = torch.device("cuda")
    rows = pot._release_seeds(torch.as_tensor(w, device=dev),
                              torch.arange(n, dtype=torch.int32, device=dev),
                              torch.as_tensor(G * msat, device=dev), seed0, nseed, 1.0,
                              t_rel=np.zeros(n))
    rows = rows.cpu().numpy()
    assert rows.shape == (nseed, 2, n, 6)
    for s in sorted({0, nseed // 2, nseed - 1}):
        pc, pf, vc, vf = oracle.release(h, w, np.zeros(n), msat, seed0 + s, src=osrc)
        for arm, (p, v) in enumerate(((pc, vc), (pf, vf))):
            ref = np.hstack([p, v])
            err = np.abs(rows[s, arm] - ref).max(0) / np.abs(ref).max(0)
            assert err.max() <= 1e-11
