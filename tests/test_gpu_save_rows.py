"""Saved rows of the fixed-step stepper on every launch path: saves at every row (the straight
code of launches that save most of their steps), the same row twice, rows before the first start,
the last row, one row among many steps, none, and rows that end early or come after a row out of
order (never reached, so left as they were).  Against the oracle's trajectory, <= 1e-11
relative."""
import numpy as np
import pytest
import torch

from test_gpu_core import bound_orbits

pytestmark = pytest.mark.gpu

G = 4.498502151469553e-12
NSTEPS = 24
SAVES = {
    "every row": list(range(NSTEPS + 1)),
    "rows twice": sorted(list(range(NSTEPS + 1)) + [0, 5, 5, 12, NSTEPS]),
    "most, ending early": list(range(2, 17)),
    "a few": [0, 9, NSTEPS],
    "last": [NSTEPS],
    "out of order": list(range(3, 16)) + [4, 20],
}


@pytest.mark.parametrize("m,n", [(0, 1), (0, 300), (7, 1), (20, 500), (64, 1), (70, 1100)])
@pytest.mark.parametrize("rows", list(SAVES))
def test_saved_rows(oracle, ssc, m, n, rows):
    from streamsculptor_amd import workloads as W
    from streamsculptor_amd.potential import PlummerClumps, Potential_Combine
    rng = np.random.default_rng(7 + m + n)
    pot, osrc, h = W.host_potential(), None, oracle.host(W.host_components())
    if m:
        pos, mass = rng.normal(scale=12.0, size=(m, 3)), 10 ** rng.uniform(6.0, 7.5, m)
        rs = rng.uniform(0.1, 0.6, m)
        pot = Potential_Combine([pot, PlummerClumps(mass, rs, pos, units=ssc.usys)],
                                units=ssc.usys)
        osrc = oracle.Sources(oracle.SRC_STATIC, gm=G * mass, rs=rs, pos=pos)
    w0 = bound_orbits(rng, n)
    start = np.sort(rng.integers(2, NSTEPS + 2, n)).astype(np.int32) if n > 1 else None
    save = SAVES[rows]
    out, ys = pot._leapfrog(w0, 0.0, 1.0, NSTEPS, start=start, save_idx=save)
    final, traj = oracle.leapfrog(h, w0, 0.0, 1.0, NSTEPS, start=start, src=osrc, traj=True)
    rel = lambda a, b: (np.linalg.norm(a - b, axis=-1) / np.linalg.norm(b, axis=-1)).max()  # noqa
    assert rel(out.cpu().numpy(), final) <= 1e-11
    reached = len(save) - 2 if rows == "out of order" else len(save)
    assert rel(ys[:reached].cpu().numpy(), traj[save[:reached]]) <= 1e-11
