"""Potential evaluation over its launch shapes: one to 64 lanes per point (the rule on the number of
points and sources), tiles of the source table with remainders, straight-line sources of which
some are outside their windows, and every combination of outputs.  Against the oracle on a sample
of the points: 1e-12 of the largest value for phi and the gradient, 1e-11 for the Hessian (the
bounds of the evaluation test)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

G = 4.498502151469553e-12


def _case(oracle, kind, m, rng):
    from streamsculptor_amd import _lib
    from streamsculptor_amd.main import Potential, SourceSet
    comps = [(1, [G * 6.8e10, 3.0, 0.28]), (2, [G * 5.4e11, 15.62])]
    src = so = None
    if m:
        gm = G * 10 ** rng.uniform(6, 8, m)
        rs = 1.62 * np.sqrt(gm / G / 1e8)
        pos = rng.normal(scale=9.0, size=(m, 3))
        if kind == "static":
            src = SourceSet(_lib.SRC_STATIC, gm=gm, rs=rs, pos=pos)
            so = oracle.Sources(oracle.SRC_STATIC, gm=gm, rs=rs, pos=pos)
        elif kind.startswith("track"):
            kk, ko = ((_lib.SRC_TRACK, oracle.SRC_TRACK) if kind == "track" else
                      (_lib.SRC_TRACK_HERNQUIST, oracle.SRC_TRACK_HERNQUIST))
            pos = np.stack([pos - 1.0, pos, pos + 1.0])
            src = SourceSet(kk, gm=gm, rs=rs, pos=pos, grid=(-50.0, 50.0))
            so = oracle.Sources(ko, gm=gm, rs=rs, pos=pos)
        else:
            kk, ko = ((_lib.SRC_LINE, oracle.SRC_LINE) if kind == "line" else
                      (_lib.SRC_LINE_HERNQUIST, oracle.SRC_LINE_HERNQUIST))
            vel, t0 = rng.normal(scale=0.2, size=(m, 3)), rng.uniform(-100, 100, m)
            kw = dict(gm=gm, rs=rs, pos=pos, vel=vel, t0=t0, t_window=rng.uniform(20, 100, m))
            src, so = SourceSet(kk, **kw), oracle.Sources(ko, **kw)

    class Pot(Potential):
        def __init__(self):
            super().__init__(None, {})

        def _kernel_components(self):
            return comps

        def _kernel_sources(self):
            return src

    return Pot(), oracle.host(comps), so


@pytest.mark.parametrize("kind,m,n", [
    ("static", 0, 5),                  # no sources
    ("static", 1, 1),                  # one lane: fewer than four sources a lane
    ("static", 15, 300),               # too few sources for 4 lanes
    ("static", 16, 8191),              # 4 lanes, from 64 narrowed by the sources
    ("line", 257, 500),                # 64 lanes, a second tile of one source
    ("hernquist", 256, 8192),          # 16 lanes, one full tile
    ("track", 255, 32767),             # 16 lanes, a tile short of one
    ("track hernquist", 64, 32768),    # 4 lanes
    ("static", 1024, 131071),          # 4 lanes, the largest table
    ("line", 300, 131072),             # one lane per point
])
def test_eval_shapes(oracle, ssc, kind, m, n):
    rng = np.random.default_rng(n + m)
    pot, h, so = _case(oracle, kind, m, rng)
    pts = rng.normal(scale=10.0, size=(n, 3))
    x = torch.as_tensor(pts, device="cuda")
    print(f"[eval] {kind} m={m} n={n}", flush=True)
    sel = np.unique(np.concatenate([[0, n - 1], rng.integers(0, n, 200)]))
    want = dict(zip(("phi", "grad", "hess"), oracle.evaluate(h, pts[sel], t=0.0, step=1, src=so)))
    tol = dict(phi=1e-12, grad=1e-12, hess=1e-11)
    for names in (("phi",), ("grad",), ("hess",), ("phi", "grad"), ("grad", "hess")):
        out = pot._eval(x, 0.0, **{"want_" + k: True for k in names})
        for k, v in zip(names, out if len(names) > 1 else (out,)):
            a, b = v.cpu().numpy()[sel].reshape(len(sel), -1), want[k].reshape(len(sel), -1)
            assert np.isfinite(v.cpu().numpy()).all()
            assert np.abs(a - b).max() <= tol[k] * np.abs(b).max(), (names, k)
