"""The adaptive responses' rows, bit for bit: final and saved rows and step counts of
ssc_perturb_dopri5 against stored ones (golden/perturb_dopri5_rows.npz, written by the kernel whose
lanes formed one host component each with the IEEE operations).  A step sequence follows the last
bits of every force, and windows of subhalos make the right-hand side jump inside steps: forms of
the host that differ in their last bits moved these rows by up to 1e-7, far above what rounding does
to one step and far below the solver's own error, which is all that a comparison with another
implementation bounds.  Hence equality.  Lane layouts: 8, 64 and 128 lanes a particle, and 256 with
one, two and four vectors a lane; hosts of three, four and six components."""
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

G = 4.498502151469553e-12
ROWS = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "perturb_dopri5_rows.npz")
CASES = [  # name, host, profile, radius block, subhalos, particles, t1
    ("groups_of_8", "three", "line", False, 3, 40, 600.0),
    ("groups_of_64", "six", "hernquist", False, 61, 4, -600.0),
    ("two_waves", "four", "hernquist", True, 37, 5, -500.0),
    ("four_waves", "three", "hernquist", True, 128, 3, -900.0),
    ("two_vectors", "three", "static", True, 150, 2, 400.0),
    ("four_vectors", "six", "line", True, 260, 2, -300.0),
]


def _host(name):
    from streamsculptor_amd import potential as P
    from streamsculptor_amd import workloads as W
    from streamsculptor_amd.main import usys
    if name == "three":
        return W.host_potential()
    disk = P.MiyamotoNagaiDisk(m=6.8e10, a=3.0, b=0.28, units=usys)
    halo = P.NFWPotential(m=5.4e11, r_s=15.62, units=usys)
    bulge = [P.HernquistPotential(m=m, r_s=r, units=usys) for m, r in ((5e9, 1.0), (1.7e9, 0.07))]
    extra = [P.PlummerPotential(m=1e10, r_s=r, units=usys) for r in (2.0, 3.5)]
    parts = [disk, *bulge, halo] if name == "four" else [halo, extra[0], disk, *bulge, extra[1]]
    return P.Potential_Combine(parts, units=usys)


def inputs(name, profile, radius, m, n, t1):
    rng = np.random.default_rng(1000 * m + n)
    r = rng.uniform(8.0, 25.0, n)
    u, v = (a / np.linalg.norm(a, axis=1, keepdims=True) for a in rng.normal(size=(2, n, 3)))
    gm = G * 10 ** rng.uniform(6, 8, m)
    d = dict(w0=np.concatenate([r[:, None] * u, 0.17 * v], 1),
             dw0=rng.normal(scale=1e-3, size=(n, m, 12 if radius else 6)),
             gm=gm, rs=1.62 * np.sqrt(gm / G / 1e8), pos=rng.normal(scale=10.0, size=(m, 3)))
    if profile != "static":
        d.update(vel=rng.normal(scale=0.2, size=(m, 3)),
                 t0=rng.uniform(min(0.0, t1), max(0.0, t1), m), t_window=rng.uniform(100, 400, m))
    return d


def solve(case, d):
    from streamsculptor_amd import _lib
    from streamsculptor_amd.fields import perturb_dopri5
    from streamsculptor_amd.main import SourceSet
    _, host, profile, radius, _, n, t1 = case
    kind = {"static": _lib.SRC_STATIC, "line": _lib.SRC_LINE,
            "hernquist": _lib.SRC_LINE_HERNQUIST}[profile]
    src = SourceSet(kind, **{k: d[k] for k in ("gm", "rs", "pos", "vel", "t0", "t_window") if k in d})
    w, dw, ys, dys, st = perturb_dopri5(
        _host(host), src, d["w0"], d["dw0"], t1, t_start=np.linspace(0.0, 0.5 * t1, n),
        ts=np.array([0.7 * t1]), with_radius=radius, rtol=1e-9, atol=1e-10, dtmin=0.01, dtmax=25.0,
        max_steps=20_000)
    return {k: v.cpu().numpy() for k, v in dict(w=w, dw=dw, ys=ys, dys=dys, stats=st).items()}


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_rows_are_the_stored_ones(ssc, case):
    z = np.load(ROWS)
    d = {k.split("/")[2]: z[k] for k in z.files if k.startswith(case[0] + "/in/")}
    print(f"[adaptive responses] {case}", flush=True)
    got = solve(case, d)
    assert (got["stats"][:, 2] == 0).all() and np.isfinite(got["dw"]).all()
    for k, v in got.items():
        np.testing.assert_array_equal(v, z[f"{case[0]}/out/{k}"], err_msg=k)
