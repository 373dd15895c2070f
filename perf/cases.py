"""Cases of the performance measurement: what a user of the framework has it do, over the sizes
and options in use.

``listed()`` gives the fixed cases and ``draw(rng)`` one more of the same ranges; a case is a dict
of plain values whose ``path`` selects one of the classes below.  Each class makes what the
user's program holds before the call (``prepare``), runs one pass through the public entry points
(``run``), states the bytes and operations that pass cannot do without (``work``) and, where it is
affordable, computes the same outputs in plain float64 torch (``exact``).
"""
import math

import numpy as np
import torch

from streamsculptor_amd import flops
from streamsculptor_amd import workloads as W

F64 = torch.float64
G = W.G
MN, NFW, HERNQUIST = 1, 2, 3
HOST = [(k, p) for k, p in W.host_components()]
MILKY_WAY = [(k, p) for k, p in W.gala_mw_components()]
# values (particles x steps x sources, ...) up to which the float64 references are formed
EXACT_PAIRS = 6e9


# ---------------------------------------------------------------------------------------------
# plain float64 references
# ---------------------------------------------------------------------------------------------
def _cat3(a, b, c):
    return torch.stack([a, b, c], -1)


def host_terms(comps, x, hess=False):
    """Potential, gradient (n, 3) and Hessian (n, 3, 3) (None unless hess) of analytic components
    ``[(kind, [G m, p1, p2])]``; the parameters may be tensors that carry gradients."""
    phi, g = 0.0, 0.0
    H = 0.0 if hess else None
    eye = torch.eye(3, dtype=F64, device=x.device)
    X, Y, Z = x.unbind(-1)
    for kind, p in comps:
        gm = p[0]
        if kind == MN:
            a, b = p[1], p[2]
            zeta = torch.sqrt(Z * Z + b * b)
            S = a + zeta
            D2 = X * X + Y * Y + S * S
            D = torch.sqrt(D2)
            phi = phi - gm / D
            q = _cat3(X, Y, Z * S / zeta)
            f = gm / (D2 * D)
            g = g + f[..., None] * q
            if hess:
                ddz = S * b * b / zeta ** 3 + Z * Z / zeta ** 2
                diag = torch.diag_embed(_cat3(torch.ones_like(ddz), torch.ones_like(ddz), ddz))
                H = H + f[..., None, None] * diag - (3.0 * f / D2)[..., None, None] * (
                    q[..., :, None] * q[..., None, :])
            continue
        if kind == NFW:
            r = torch.sqrt((x * x).sum(-1))
            rp = r + p[1]
            L = torch.log1p(r / p[1])
            phi = phi - gm * L / r
            d1 = gm * (L / (r * r) - 1.0 / (r * rp))
            d2 = gm * (1.0 / (r * r * rp) - 2.0 * L / r ** 3 + (2.0 * r + p[1]) / (r * rp) ** 2)
        else:
            r = torch.sqrt((x * x).sum(-1))
            rc = r + p[1]
            phi = phi - gm / rc
            d1 = gm / (rc * rc)
            d2 = -2.0 * gm / rc ** 3
        d1r = d1 / r
        g = g + d1r[..., None] * x
        if hess:
            H = H + d1r[..., None, None] * eye + ((d2 - d1r) / (r * r))[..., None, None] * (
                x[..., :, None] * x[..., None, :])
    return phi, g, H


def plummer_terms(x, pos, gm, rs, hess=False):
    """The same for a sum of Plummer sources at pos (M, 3) or one set per row (n, M, 3)."""
    d = x[..., None, :] - pos
    s2 = (d * d).sum(-1) + rs * rs
    i1 = s2.rsqrt()
    f = gm * i1 * i1 * i1
    phi = -(gm * i1).sum(-1)
    g = (f[..., None] * d).sum(-2)
    H = None
    if hess:
        k = -3.0 * f * i1 * i1
        H = f.sum(-1)[..., None, None] * torch.eye(3, dtype=F64, device=x.device)
        H = H + torch.matmul((k[..., None] * d).transpose(-1, -2).contiguous(), d)
    return phi, g, H


def plummer_chunked(x, pos, gm, rs, hess=False, pairs=1 << 25):
    step = max(1, pairs // max(1, pos.shape[0]))
    out = [plummer_terms(x[i:i + step], pos, gm, rs, hess) for i in range(0, x.shape[0], step)]
    return [None if o[0] is None else torch.cat(o) for o in zip(*out)]


def leapfrog(accel, w, start, dt, nsteps, keep=False):
    """Kick-drift-kick on rows k = 0..nsteps; orbit i moves from row start[i].  accel(x, k)."""
    x, v = w[:, :3], w[:, 3:]
    rows = [torch.cat([x, v], 1)] if keep else None
    a = accel(x, 0)
    for k in range(nsteps):
        on = None if start is None else (start <= k)[:, None]
        vh = v + 0.5 * dt * a
        xn = x + dt * vh
        if on is not None:
            xn = torch.where(on, xn, x)
        a = accel(xn, k + 1)
        vn = vh + 0.5 * dt * a
        v = vn if on is None else torch.where(on, vn, v)
        x = xn
        if keep:
            rows.append(torch.cat([x, v], 1))
    return torch.stack(rows) if keep else torch.cat([x, v], 1)


DP_A = ((1 / 5,), (3 / 40, 9 / 40), (44 / 45, -56 / 15, 32 / 9),
        (19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729),
        (9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656),
        (35 / 384, 0.0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84))
DP_C = (1 / 5, 3 / 10, 4 / 5, 8 / 9, 1.0, 1.0)
DP_E = (71 / 57600, 0.0, -71 / 16695, 71 / 1920, -17253 / 339200, 22 / 525, -1 / 40)
DP_M = (6025192743 / 30085553152 / 2, 0.0, 51252292925 / 65400821598 / 2,
        -2691868925 / 45128329728 / 2, 187940372067 / 1594534317056 / 2,
        -1776094331 / 19743644256 / 2, 11237099 / 235043384 / 2)


def _sum(weights, ks):
    return sum(w * k for w, k in zip(weights, ks) if w != 0.0)


def dopri5(f, y, t0, t1, ts=None, rtol=1e-7, atol=1e-7, dtmin=0.3, max_steps=10_000):
    """Dormand-Prince 5(4) of n independent systems y (n, N) from t0 (n,) to t1, each with its
    own integral step controller; f(t (n,), y, rows) with rows the systems' indices.  Saves at
    ts (k,), monotone in the direction of integration, by the quartic dense output.  Returns
    (final rows, saved rows (n, k, N) or None)."""
    n, N = y.shape
    dev = y.device
    dirn = torch.where(t1 - t0 >= 0, 1.0, -1.0).to(F64)
    tau, end = dirn * t0, dirn * t1
    y = y.clone()
    save = None if ts is None else torch.full((n, len(ts), N), float("nan"), dtype=F64, device=dev)
    taus = None if ts is None else dirn[:, None] * ts[None, :]
    if ts is not None:
        at = taus == tau[:, None]
        save[at] = y[:, None, :].expand(n, len(ts), N)[at]

    def rhs(tt, yy, rows):
        return dirn[rows, None] * f(dirn[rows] * tt, yy, rows)

    def rms(u):
        return torch.sqrt((u * u).mean(1))

    rows = torch.nonzero(tau < end).flatten()
    k0 = torch.zeros_like(y)
    k0[rows] = rhs(tau[rows], y[rows], rows)
    sc = atol + y.abs() * rtol
    d0, d1 = rms(y / sc), rms(k0 / sc)
    h0 = torch.where((d0 < 1e-5) | (d1 < 1e-5), torch.full_like(d0, 1e-6), 0.01 * d0 / d1)
    f1 = torch.zeros_like(y)
    f1[rows] = rhs((tau + h0)[rows], (y + h0[:, None] * k0)[rows], rows)
    md = torch.maximum(d1, rms((f1 - k0) / sc) / h0)
    h = torch.minimum(100.0 * h0, torch.where(md <= 1e-15, torch.clamp(h0 * 1e-3, min=1e-6),
                                              (0.01 / md) ** 0.2))
    floor = h <= dtmin
    nxt = torch.minimum(tau + torch.clamp(h, min=dtmin), end)
    for _ in range(max_steps):
        rows = torch.nonzero(tau < end).flatten()
        if rows.numel() == 0:
            break
        t, yr, hr = tau[rows], y[rows], (nxt - tau)[rows]
        hc = hr[:, None]
        ks = [k0[rows]]
        for a, c in zip(DP_A, DP_C):
            yn = yr + hc * _sum(a, ks)
            ks.append(rhs(t + c * hr, yn, rows))
        e = rms(hc * _sum(DP_E, ks) / (atol + rtol * torch.maximum(yr.abs(), yn.abs())))
        ok = (e < 1.0) | floor[rows]
        fac = torch.clamp(0.9 * (1.0 / e) ** 0.2, max=10.0)
        new = hr * torch.maximum(fac, torch.where(ok, 1.0, 0.2).to(F64))
        floor[rows] = new <= dtmin
        new = torch.clamp(new, min=dtmin)
        if ts is not None:
            tr, tn = taus[rows], (t + hr)[:, None]
            hit = (tr > t[:, None]) & (tr <= tn) & ok[:, None]
            if bool(hit.any()):
                ym = yr + hc * _sum(DP_M, ks)
                F0, F1 = hc * ks[0], hc * ks[6]
                D1, D2, D3 = yn - yr - F0, F1 - F0, ym - yr - 0.5 * F0
                a4 = 2.0 * D2 - 8.0 * D1 + 16.0 * D3
                b3 = D2 - 2.0 * D1 - 2.0 * a4
                c2 = D1 - a4 - b3
                r, j = torch.nonzero(hit, as_tuple=True)
                s = ((tr[r, j] - t[r]) / hr[r])[:, None]
                v = yr[r] + s * (F0[r] + s * (c2[r] + s * (b3[r] + s * a4[r])))
                save[rows[r], j] = torch.where(s == 1.0, yn[r], v)
        m = rows[ok]
        y[m], k0[m], tau[m] = yn[ok], ks[6][ok], (t + hr)[ok]
        t1n = tau[rows] + new
        near = t1n > end[rows] - 1e-10
        last = torch.where(ok, end[rows], tau[rows] + 0.5 * (end[rows] - tau[rows]))
        nxt[rows] = torch.where(near, last, t1n)
    return y, save


M32 = 0xFFFFFFFF


def threefry(k0, k1, x0, x1):
    """Threefry-2x32 with 20 rounds on Python integers."""
    ks = (k0, k1, k0 ^ k1 ^ 0x1BD11BDA)
    a, b = (x0 + k0) & M32, (x1 + k1) & M32
    for blk in range(5):
        for r in ((13, 15, 26, 6), (17, 29, 16, 24))[blk & 1]:
            a = (a + b) & M32
            b = (((b << r) | (b >> (32 - r))) & M32) ^ a
        a = (a + ks[(blk + 1) % 3]) & M32
        b = (b + ks[(blk + 2) % 3] + blk + 1) & M32
    return a, b


def release_keys(seed):
    """The four per-release key factors of a release seed."""
    hi, lo = (seed >> 32) & M32, seed & M32
    a, b = threefry(hi, lo, 0, 2), threefry(hi, lo, 1, 3)
    mult = ((1 << 32) % 1000) ** 2 % 1000
    out = []
    for j in range(4):
        h, l = (threefry(a[i], b[i], j, 5 + j) for i in (0, 1))
        h, l = (h[0] << 32) | h[1], (l[0] << 32) | l[1]
        out.append(((h % 1000) * mult + l % 1000) % 1000)
    return out


def release_normals(idx, seed, dev):
    """(len(idx), 4) Gaussian multipliers of the releases ``idx``."""
    out = np.empty((len(idx), 4))
    keys = release_keys(seed)
    for i, r in enumerate(idx):
        for k, key in enumerate(keys):
            s = int(r) * key
            hi, lo = threefry((s >> 32) & M32, s & M32, 0, 1)
            bits = (((hi << 32) | lo) >> 12) | 0x3FF0000000000000
            out[i, k] = np.array([bits], dtype=np.uint64).view(np.float64)[0] - 1.0
    low = -0.99999999999999988898
    u = torch.as_tensor(out, dtype=F64, device=dev) * 2.0 + low
    return math.sqrt(2.0) * torch.erfinv(torch.clamp(u, min=low))


def release(w, H, msat, z):
    """Spray release rows (n, 2, 6) (leading, trailing) of progenitor rows w in a potential with
    Hessian H there."""
    x, v = w[:, :3], w[:, 3:]
    r = torch.sqrt((x * x).sum(1, keepdim=True))
    rh = x / r
    d2 = (rh[:, None, :] * H * rh[:, :, None]).sum((1, 2))
    L = torch.linalg.cross(x, v, dim=1)
    Ln = torch.sqrt((L * L).sum(1))
    om = Ln / r[:, 0] ** 2
    rt = (G * msat / (om * om - d2)) ** (1.0 / 3.0)
    zh = L / Ln[:, None]
    pv = v - (v * rh).sum(1, keepdim=True) * rh
    ph = pv / torch.sqrt((pv * pv).sum(1, keepdim=True))
    kr = 2.0 + 0.4 * z[:, 0]
    kp = kr * (0.3 + 0.4 * z[:, 1])
    dp = (kr * rt)[:, None] * rh + (0.5 * z[:, 2] * rt)[:, None] * zh
    dv = (om * rt)[:, None] * (kp[:, None] * ph + (0.5 * z[:, 3])[:, None] * zh)
    return torch.stack([torch.cat([x - dp, v - dv], 1), torch.cat([x + dp, v + dv], 1)], 1)


def spray_rows(prog, H, msat, per_step, seed):
    """Rows and start rows of the many-particle spray: per_step particles at every release row
    (prog (T, 6)), seeds and arms in the framework's order."""
    T = prog.shape[0]
    nseed = (per_step + 1) // 2
    table = torch.stack([release(prog, H, msat, release_normals(range(T), seed + s, prog.device))
                         for s in range(nseed)])                       # (seed, T, arm, 6)
    lay = np.array(W.spray_layout(per_step))[np.arange(T) % 2]         # (T, per_step, 2)
    rel = torch.arange(T, device=prog.device).repeat_interleave(per_step)
    sel = torch.as_tensor(lay.reshape(-1, 2), device=prog.device)
    return table[sel[:, 0], rel, sel[:, 1]], rel


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
def gpu(a):
    return torch.as_tensor(np.asarray(a), dtype=F64, device="cuda")


def jitter(row, seed, scale=0.03):
    """A progenitor row near ``row``: the same kind of orbit for every seed."""
    return np.asarray(row) * (1.0 + scale * np.random.default_rng(seed).uniform(-1, 1, 6))


def back_rows(comps, row, dt, nsteps):
    """Rows (nsteps + 1, 6) of one orbit walked by dt from ``row`` (plain Python leapfrog)."""
    def acc(x, y, z):
        ax = ay = az = 0.0
        for kind, p in comps:
            if kind == MN:
                zeta = math.sqrt(z * z + p[2] * p[2])
                S = p[1] + zeta
                f = p[0] / (x * x + y * y + S * S) ** 1.5
                ax, ay, az = ax - f * x, ay - f * y, az - f * z * S / zeta
                continue
            r = math.sqrt(x * x + y * y + z * z)
            if kind == NFW:
                f = p[0] * (math.log1p(r / p[1]) / r - 1.0 / (r + p[1])) / (r * r)
            else:
                f = p[0] / (r * (r + p[1]) ** 2)
            ax, ay, az = ax - f * x, ay - f * y, az - f * z
        return ax, ay, az
    x, y, z, u, v, w = (float(c) for c in row)
    out = [(x, y, z, u, v, w)]
    ax, ay, az = acc(x, y, z)
    for _ in range(nsteps):
        u, v, w = u + 0.5 * dt * ax, v + 0.5 * dt * ay, w + 0.5 * dt * az
        x, y, z = x + dt * u, y + dt * v, z + dt * w
        ax, ay, az = acc(x, y, z)
        u, v, w = u + 0.5 * dt * ax, v + 0.5 * dt * ay, w + 0.5 * dt * az
        out.append((x, y, z, u, v, w))
    return np.array(out)


def orbits(n, seed, lo=8.0, hi=18.0):
    """n bound rows: isotropic positions between lo and hi kpc, mostly tangential speeds."""
    rng = np.random.default_rng(seed)
    u = rng.normal(size=(n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    t = np.cross(u, rng.normal(size=(n, 3)))
    t /= np.linalg.norm(t, axis=1, keepdims=True)
    return np.hstack([rng.uniform(lo, hi, n)[:, None] * u,
                      rng.uniform(0.15, 0.21, n)[:, None] * t
                      + rng.normal(scale=0.01, size=(n, 3))])


def potential(name):
    from streamsculptor_amd.main import usys
    from streamsculptor_amd.potential import GalaMilkyWayPotential
    return W.host_potential() if name == "host" else GalaMilkyWayPotential(units=usys)


def components(name):
    return HOST if name == "host" else MILKY_WAY


def with_clumps(case, seed):
    """Host + static clumps, and the clumps alone."""
    from streamsculptor_amd.main import usys
    from streamsculptor_amd.potential import PlummerClumps, Potential_Combine
    host = W.host_potential()
    pos, m, rs = W.clump_table(n=case["sources"], seed=seed)
    clumps = PlummerClumps(m, rs, pos, units=usys)
    return host, clumps, Potential_Combine([host, clumps], units=usys)


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# ---------------------------------------------------------------------------------------------
# the paths
# ---------------------------------------------------------------------------------------------
class Orbit:
    """``integrate_orbit`` of one orbit or a batch with saved rows: the smallest call, bound by
    latency and launches."""

    @staticmethod
    def draw(rng):
        return dict(n=log_int(rng, 1, 3000), age=rng.randint(500, 4000),
                    saves=log_int(rng, 2, 1000), solver=rng.choice(["dopri5", "leapfrog"]),
                    potential=rng.choice(["host", "milky way"]))

    @staticmethod
    def times(case):
        k = np.unique(np.rint(np.linspace(0, case["age"], case["saves"])))
        return k - case["age"]

    @staticmethod
    def prepare(case, seed):
        w0 = orbits(case["n"], seed)
        return dict(pot=potential(case["potential"]), w0=gpu(w0[0] if case["n"] == 1 else w0),
                    ts=Orbit.times(case), case=case)

    @staticmethod
    def run(s):
        return s["pot"].integrate_orbit(w0=s["w0"], ts=s["ts"], solver=s["case"]["solver"],
                                        dt0=1.0 if s["case"]["solver"] == "leapfrog" else None).ys

    @staticmethod
    def work(case):
        # the adaptive solver takes about one step per 5 Myr here
        per = flops.plain() * case["age"] if case["solver"] == "leapfrog" else (
            flops.dopri5_step() * case["age"] / 5)
        return dict(bytes=48.0 * case["n"] * (1 + case["saves"]), flops=per * case["n"])

    @staticmethod
    def exact(case, seed):
        w0, ts, comps = gpu(orbits(case["n"], seed)), Orbit.times(case), components(case["potential"])
        if case["solver"] == "leapfrog":
            rows = leapfrog(lambda x, k: -host_terms(comps, x)[1], w0, None, 1.0,
                            int(case["age"]), keep=True)
            ys = rows[torch.as_tensor(ts + case["age"], device="cuda").long()].permute(1, 0, 2)
        else:
            _, ys = dopri5(_orbit_rhs(comps), w0, torch.full((case["n"],), float(ts[0]), dtype=F64,
                                                            device="cuda"), 0.0, gpu(ts))
        return ys[0] if case["n"] == 1 else ys


def _orbit_rhs(comps, src=None):
    def f(t, y, rows):
        g = host_terms(comps, y[:, :3])[1]
        if src is not None:
            g = g + src(t, y[:, :3], rows)
        return torch.cat([y[:, 3:], -g], 1)
    return f


class Evaluate:
    """Potential, gradient and Hessian of a (clumpy) halo at many points: maps, labels for the
    learned force, tidal fields."""

    @staticmethod
    def draw(rng):
        return dict(n=log_int(rng, 500, 600000), sources=rng.choice([0, log_int(rng, 16, 1024)]))

    @staticmethod
    def points(case, seed):
        g = np.random.default_rng(seed)
        u = g.normal(size=(case["n"], 3))
        return g.uniform(1.0, 40.0, (case["n"], 1)) * u / np.linalg.norm(u, axis=1, keepdims=True)

    @staticmethod
    def prepare(case, seed):
        host, _, pot = with_clumps(case, seed) if case["sources"] else (W.host_potential(),) * 3
        return dict(pot=pot, x=gpu(Evaluate.points(case, seed)))

    @staticmethod
    def run(s):
        return dict(phi=s["pot"].potential(s["x"], 0.0), grad=s["pot"].gradient(s["x"], 0.0),
                    hess=s["pot"].jacobian_force(s["x"], 0.0))

    @staticmethod
    def work(case):
        # potential 11, gradient 18 and Hessian 30 operations per source; the host's likewise
        return dict(bytes=case["n"] * 8.0 * (3 + 1 + 3 + 9) + 40.0 * case["sources"],
                    flops=case["n"] * (190.0 + (11 + 18 + 30) * case["sources"]))

    @staticmethod
    def exact(case, seed):
        x = gpu(Evaluate.points(case, seed))
        out = host_terms(HOST, x, True)
        if case["sources"]:
            pos, m, rs = W.clump_table(n=case["sources"], seed=seed)
            out = [a + b for a, b in zip(out, plummer_chunked(x, gpu(pos), gpu(G * m), gpu(rs), True))]
        return dict(phi=out[0], grad=out[1], hess=out[2])


class Stream:
    """``gen_stream_vmapped``: the spray stream with two particles per release step, fixed-step or
    adaptive."""

    @staticmethod
    def draw(rng):
        return dict(steps=log_int(rng, 120, 5000), solver=rng.choice(["dopri5", "leapfrog"]),
                    potential=rng.choice(["host", "milky way"]))

    @staticmethod
    def times(case):
        return W.release_times(case["steps"]) if case["solver"] == "leapfrog" else np.linspace(
            -3000.0, 0.0, case["steps"] + 1)

    @staticmethod
    def first_row(case, seed):
        return back_rows(components(case["potential"]), jitter(W.PROG_TODAY, seed), -1.0,
                         int(-Stream.times(case)[0]))[-1]

    @staticmethod
    def prepare(case, seed):
        return dict(pot=potential(case["potential"]), ts=Stream.times(case), seed=seed % 1000,
                    w0=gpu(Stream.first_row(case, seed)), solver=case["solver"])

    @staticmethod
    def run(s):
        return s["pot"].gen_stream_vmapped(ts=s["ts"], prog_w0=s["w0"], Msat=W.MSAT,
                                           seed_num=s["seed"], solver=s["solver"],
                                           dt0=W.DT if s["solver"] == "leapfrog" else None)

    @staticmethod
    def work(case):
        n = 2 * case["steps"]
        per = flops.plain() * case["steps"] / 2 if case["solver"] == "leapfrog" else (
            flops.dopri5_step() * 1500 / 5)
        return dict(bytes=96.0 * n, flops=per * n)

    @staticmethod
    def exact(case, seed):
        comps, ts = components(case["potential"]), gpu(Stream.times(case))
        w0, T = gpu(Stream.first_row(case, seed))[None], case["steps"]
        z = release_normals(range(T), seed % 1000, "cuda")
        if case["solver"] == "leapfrog":
            prog = leapfrog(lambda x, k: -host_terms(comps, x)[1], w0, None, W.DT, T, keep=True)[:, 0]
        else:
            prog = dopri5(_orbit_rhs(comps), w0, ts[:1], 0.0, ts)[1][0]
        rows = release(prog[:T], host_terms(comps, prog[:T, :3], True)[2], W.MSAT, z).reshape(-1, 6)
        if case["solver"] == "leapfrog":
            start = torch.arange(T, device="cuda").repeat_interleave(2)
            out = leapfrog(lambda x, k: -host_terms(comps, x)[1], rows, start, W.DT, T)
        else:
            out = dopri5(_orbit_rhs(comps), rows, ts[:T].repeat_interleave(2), 0.0)[0]
        return out[0::2], out[1::2]


class Batch:
    """Many perturbed GD-1-like streams at once with the adaptive solver, one straight-line
    subhalo each: the progenitors back, then ``gen_stream_batch_with_pert``."""
    TOL = dict(rtol=1e-6, atol=1e-6, dtmin=0.05, max_steps=10_000)

    @staticmethod
    def draw(rng):
        strip = log_int(rng, 60, 2000)
        return dict(sims=log_int(rng, 1, 700), strip=strip)

    @staticmethod
    def inputs(case, seed):
        back = back_rows(MILKY_WAY, jitter(W.GD1_TODAY, seed, 0.01), -1.0, int(W.GD1_AGE))
        pr = W.gd1_subhalo_prior(case["sims"], seed=seed)
        k = np.clip(np.rint(pr["t_impact"]).astype(np.int64), 1, int(W.GD1_AGE))
        return back[0], W.gd1_ts(case["strip"]), dict(
            m=pr["m"], a=pr["a"], x0=back[k, :3] + pr["b"][:, None] * pr["dir_b"],
            v=back[k, 3:] + pr["v"][:, None] * pr["dir_v"], t=-k.astype(np.float64))

    @staticmethod
    def prepare(case, seed):
        from streamsculptor_amd.batch import SubhaloLineBatch
        from streamsculptor_amd.main import usys
        today, ts, p = Batch.inputs(case, seed)
        batch = SubhaloLineBatch(p["m"][:, None], p["a"][:, None], p["x0"][:, None],
                                 p["v"][:, None], p["t"][:, None],
                                 np.full((case["sims"], 1), 100.0), units=usys)
        return dict(pot=potential("milky way"), batch=batch, today=gpu(today), ts=ts,
                    seed=seed % 1000)

    @staticmethod
    def run(s):
        from streamsculptor_amd.batch import gen_stream_batch_with_pert, integrate_orbit_batch
        ic = integrate_orbit_batch(s["pot"], s["batch"], s["today"], ts=[-W.GD1_AGE], t0=0.0,
                                   t1=-W.GD1_AGE)[:, 0]
        return gen_stream_batch_with_pert(s["pot"], s["batch"], s["ts"], ic, W.MSAT, s["seed"],
                                          **Batch.TOL)

    @staticmethod
    def work(case):
        # about 90 accepted and 35 rejected steps an orbit
        n = 2.0 * case["sims"] * case["strip"]
        return dict(bytes=104.0 * n, flops=n * 125 * flops.dopri5_step(
            flops.HOST_GRAD + flops.HERNQUIST_GRAD, 0))

    @staticmethod
    def exact(case, seed):
        # orbits near a subhalo follow the last bits of every force: no value to compare with
        return None


class Live:
    """``spray_stream`` with live subhalos: direct sums over sources on tracks of their own."""

    @staticmethod
    def draw(rng):
        return dict(steps=log_int(rng, 250, 4000), per_step=log_int(rng, 1, 25),
                    sources=log_int(rng, 5, 64))

    @staticmethod
    def inputs(case, seed):
        sub, m, rs = W.subhalo_ics(n=case["sources"], seed=seed)
        return (back_rows(HOST, jitter(W.PROG_TODAY, seed), -1.0, case["steps"])[-1], sub, m, rs,
                W.release_times(case["steps"]))

    @staticmethod
    def prepare(case, seed):
        from streamsculptor_amd.main import usys
        from streamsculptor_amd.potential import LiveSubhaloPotential, Potential_Combine
        w0, sub, m, rs, ts = Live.inputs(case, seed)
        host = W.host_potential()
        live = LiveSubhaloPotential.from_orbits(host, sub, m, rs, float(ts[0]), W.DT, case["steps"])
        return dict(host=host, live=live, pot=Potential_Combine([host, live], units=usys), ts=ts,
                    w0=gpu(w0), seed=seed % 1000, case=case)

    @staticmethod
    def run(s):
        from streamsculptor_amd.streams import spray_stream
        return spray_stream(s["pot"], s["host"], s["ts"], s["w0"], W.MSAT, s["seed"],
                            s["case"]["per_step"], W.DT)

    @staticmethod
    def work(case):
        return dict(bytes=96.0 * case["steps"] * case["per_step"]
                    + 24.0 * (case["steps"] + 1) * case["sources"],
                    flops=float(W.particle_steps(case["per_step"], case["steps"]))
                    * flops.plain(case["sources"]))

    @staticmethod
    def particles(case, seed):
        """(rows, start rows, subhalo tracks, G m, r_s) of the float64 reference."""
        w0, sub, m, rs, _ = Live.inputs(case, seed)
        T, gm, rs = case["steps"], gpu(G * m), gpu(rs)
        host = lambda x, k: -host_terms(HOST, x)[1]  # noqa: E731
        track = leapfrog(host, gpu(sub), None, W.DT, T, keep=True)[..., :3].contiguous()
        full = lambda x, k: host(x, k) - plummer_terms(x, track[k], gm, rs)[1]  # noqa: E731
        prog = leapfrog(full, gpu(w0)[None], None, W.DT, T, keep=True)[:T, 0]
        rows, start = spray_rows(prog, host_terms(HOST, prog[:, :3], True)[2], W.MSAT,
                                 case["per_step"], seed % 1000)
        return rows, start, full, track, gm, rs

    @staticmethod
    def exact(case, seed):
        if case["steps"] ** 2 * case["per_step"] * case["sources"] > EXACT_PAIRS:
            return None
        rows, start, full, *_ = Live.particles(case, seed)
        return leapfrog(full, rows, start, W.DT, case["steps"])


class Clumps:
    """``spray_stream`` in a clumpy halo: direct sums over static clumps."""

    @staticmethod
    def draw(rng):
        steps, per_step = log_int(rng, 250, 4000), log_int(rng, 2, 100)
        return dict(steps=steps, per_step=per_step, sources=log_int(rng, 40, 512))

    @staticmethod
    def prepare(case, seed):
        _, _, pot = with_clumps(case, seed)
        return dict(pot=pot, ts=W.release_times(case["steps"]), seed=seed % 1000, case=case,
                    w0=gpu(back_rows(HOST, jitter(W.PROG_TODAY, seed), -1.0, case["steps"])[-1]))

    @staticmethod
    def run(s):
        from streamsculptor_amd.streams import spray_stream
        return spray_stream(s["pot"], s["pot"], s["ts"], s["w0"], W.MSAT, s["seed"],
                            s["case"]["per_step"], W.DT)

    @staticmethod
    def work(case):
        return dict(bytes=96.0 * case["steps"] * case["per_step"],
                    flops=float(W.particle_steps(case["per_step"], case["steps"]))
                    * flops.plain(case["sources"]))

    @staticmethod
    def exact(case, seed):
        if case["steps"] ** 2 * case["per_step"] * case["sources"] > EXACT_PAIRS:
            return None
        pos, m, rs = W.clump_table(n=case["sources"], seed=seed)
        pos, gm, rs = gpu(pos), gpu(G * m), gpu(rs)
        acc = lambda x, k: -host_terms(HOST, x)[1] - plummer_terms(x, pos, gm, rs)[1]  # noqa: E731
        w0 = gpu(back_rows(HOST, jitter(W.PROG_TODAY, seed), -1.0, case["steps"])[-1])[None]
        prog = leapfrog(acc, w0, None, W.DT, case["steps"], keep=True)[:-1, 0]
        H = (host_terms(HOST, prog[:, :3], True)[2]
             + plummer_terms(prog[:, :3], pos, gm, rs, True)[2])
        rows, start = spray_rows(prog, H, W.MSAT, case["per_step"], seed % 1000)
        return leapfrog(acc, rows, start, W.DT, case["steps"])


class Responses:
    """Fixed-step first-order responses of a spray stream to subhalos on their own orbits:
    releases in the host, then ``perturb_leapfrog`` of every particle."""

    @staticmethod
    def draw(rng):
        return dict(steps=log_int(rng, 250, 4000), per_step=log_int(rng, 1, 20),
                    sources=log_int(rng, 5, 64), radius=rng.random() < 0.3)

    @staticmethod
    def prepare(case, seed):
        s = Live.prepare(case, seed)
        s["src"] = s["live"]._kernel_sources()
        return s

    @staticmethod
    def run(s):
        from streamsculptor_amd.fields import perturb_leapfrog
        from streamsculptor_amd.streams import spray_particles
        w0, start, _, (t0, dt, nsteps, _) = spray_particles(
            s["host"], s["host"], s["ts"], s["w0"], W.MSAT, s["seed"], s["case"]["per_step"], W.DT)
        return perturb_leapfrog(s["host"], s["src"], w0, None, start, t0, dt, nsteps,
                                s["case"]["radius"])

    @staticmethod
    def work(case):
        n = case["steps"] * case["per_step"]
        d = 2 if case["radius"] else 1
        return dict(bytes=n * (96.0 + 48.0 * d * case["sources"])
                    + 24.0 * (case["steps"] + 1) * case["sources"],
                    flops=float(W.particle_steps(case["per_step"], case["steps"]))
                    * flops.responses(d * case["sources"]))

    @staticmethod
    def exact(case, seed):
        if case["steps"] ** 2 * case["per_step"] * case["sources"] > EXACT_PAIRS / 6:
            return None
        w0, sub, m, rs, _ = Live.inputs(case, seed)
        T, gm, rs, dt = case["steps"], gpu(G * m), gpu(rs), W.DT
        host = lambda x, k: -host_terms(HOST, x)[1]  # noqa: E731
        track = leapfrog(host, gpu(sub), None, dt, T, keep=True)[..., :3]
        prog = leapfrog(host, gpu(w0)[None], None, dt, T, keep=True)[:T, 0]
        rows, start = spray_rows(prog, host_terms(HOST, prog[:, :3], True)[2], W.MSAT,
                                 case["per_step"], seed % 1000)
        x, v = rows[:, :3], rows[:, 3:]
        blocks = 2 if case["radius"] else 1
        n, M = x.shape[0], gm.shape[0]
        dx = torch.zeros(blocks, n, M, 3, dtype=F64, device="cuda")
        dv = torch.zeros_like(dx)

        def forces(k):
            _, g, H = host_terms(HOST, x, True)
            d = x[:, None, :] - track[k]
            s2 = (d * d).sum(-1) + rs * rs
            f = gm * s2 ** -1.5
            src = [f[..., None] * d]
            if blocks == 2:
                src.append((-3.0 * rs * f / s2)[..., None] * d)
            Ht = H[None, :, None]
            return -g, -torch.stack(src) - (Ht * dx[..., None, :]).sum(-1)

        a, da = forces(0)
        for k in range(T):
            on = (start <= k)[:, None]
            h = torch.where(on, 0.5 * dt, 0.0)
            v, dv = v + h * a, dv + h[:, None] * da
            x, dx = x + 2.0 * h * v, dx + 2.0 * h[:, None] * dv
            a, da = forces(k + 1)
            v, dv = v + h * a, dv + h[:, None] * da
        return torch.cat([x, v], 1), torch.cat([t for b in range(blocks) for t in (dx[b], dv[b])], -1)


class Derivs:
    """One batch of the adaptive derivative production: the progenitor's backward responses and
    every particle's response solve to straight-line subhalos, one controller per particle."""
    TOL = dict(rtol=1e-8, atol=1e-8, dtmin=0.01, max_steps=100_000)

    @staticmethod
    def draw(rng):
        return dict(steps=log_int(rng, 60, 1000), sources=log_int(rng, 3, 128),
                    profile=rng.choice(["hernquist", "plummer"]))

    @staticmethod
    def inputs(case, seed):
        rng = np.random.default_rng(seed)
        T, m = case["steps"], case["sources"]
        ts = np.linspace(-3000.0, 0.0, T + 1)
        rows = back_rows(HOST, jitter(W.PROG_TODAY, seed), -1.0, 3000)[::-1]
        k = rng.integers(750, 3000, m)
        mass = 10 ** rng.uniform(6.0, 8.0, m)
        rs = 1.05 * np.sqrt(mass / 1e8)
        u = rng.normal(size=(m, 3))
        u /= np.linalg.norm(u, axis=1, keepdims=True)
        x0 = rows[k, :3] + rng.uniform(0.0, 5.0, m)[:, None] * rs[:, None] * u
        v = rows[k, 3:] + rng.normal(scale=0.15, size=(m, 3))
        return ts, rows[0].copy(), (mass, rs, x0, v, k - 3000.0, np.full(m, 150.0))

    @staticmethod
    def prepare(case, seed):
        from streamsculptor_amd.main import usys
        from streamsculptor_amd.perturbative import BaseStreamModel
        from streamsculptor_amd.potential import (HernquistPotential, PlummerPotential,
                                                  SubhaloLinePotentialCustom_dRadius_fromFunc,
                                                  SubhaloLinePotentialCustom_fromFunc)
        from streamsculptor_amd.solvers import Dopri5
        ts, w0, p = Derivs.inputs(case, seed)
        base = W.host_potential()
        func = HernquistPotential if case["profile"] == "hernquist" else PlummerPotential
        return dict(base=base, bs=BaseStreamModel(base, w0, ts, W.MSAT, seed % 1000, solver=Dopri5(),
                                                  rtol=1e-8, atol=1e-8, dtmin=0.01),
                    pert=SubhaloLinePotentialCustom_fromFunc(func, *p, units=usys),
                    struct=SubhaloLinePotentialCustom_dRadius_fromFunc(func, *p, units=usys))

    @staticmethod
    def run(s):
        from streamsculptor_amd.perturbative import GenerateMassRadiusPerturbation
        gen = GenerateMassRadiusPerturbation(s["base"], s["pert"], s["struct"],
                                             BaseStreamModel=s["bs"], **Derivs.TOL)
        return gen.compute_perturbation_OTF(**Derivs.TOL)

    @staticmethod
    def work(case):
        # about 700 steps over a particle's mean life of 1500 Myr
        n = 2.0 * case["steps"]
        return dict(bytes=n * (96.0 + 192.0 * case["sources"]),
                    flops=n * 700 * flops.perturb_dopri5_step(2 * case["sources"]))

    @staticmethod
    def exact(case, seed):
        if case["steps"] * case["sources"] > 10000:
            return None
        T, m = case["steps"], case["sources"]
        ts_np, w0, p = Derivs.inputs(case, seed)
        ts = gpu(ts_np)
        mass, rs, x0, v, tc, tw = (gpu(a) for a in p)
        gm = G * mass
        prog = dopri5(_orbit_rhs(HOST), gpu(w0)[None], ts[:1], 0.0, ts, rtol=1e-8, atol=1e-8,
                      dtmin=0.01)[1][0]

        def f(t, y, rows):
            n = y.shape[0]
            _, g, H = host_terms(HOST, y[:, :3], True)
            q = y[:, 6:].reshape(n, m, 2, 2, 3)                       # block, (x, v)
            dt = t[:, None] - tc
            d = y[:, None, :3] - (x0 + v * dt[..., None])
            r2 = (d * d).sum(-1)
            if case["profile"] == "hernquist":
                r = torch.sqrt(r2)
                c = gm / (r * (r + rs) ** 2)
                cr = -2.0 * c / (r + rs)
            else:
                s2 = r2 + rs * rs
                c = gm * s2 ** -1.5
                cr = -3.0 * rs * c / s2
            on = (dt.abs() < tw).to(F64)
            src = torch.stack([c * on, cr * on], -1)[..., None] * d[:, :, None, :]
            acc = -src - (H[:, None, None] * q[:, :, :, 0, None, :]).sum(-1)
            dq = torch.stack([q[:, :, :, 1], acc], 3)
            return torch.cat([y[:, 3:6], -g, dq.reshape(n, -1)], 1)

        tol = dict(Derivs.TOL)
        y0 = torch.cat([prog[-1], torch.zeros(12 * m, dtype=F64, device="cuda")])[None]
        back = dopri5(f, y0, ts[-1:], float(ts_np[0]), torch.flip(ts, [0]), **tol)[1][0]
        resp = torch.flip(back, [0])[:, 6:].reshape(T + 1, m, 2, 6)
        w = prog.detach().requires_grad_(True)
        rel = release(w, host_terms(HOST, w[:, :3], True)[2], W.MSAT,
                      release_normals(range(T + 1), seed % 1000, "cuda"))
        y0 = []
        for arm in range(2):
            J = torch.stack([torch.autograd.grad(rel[:, arm, c].sum(), w, retain_graph=True)[0]
                             for c in range(6)], 1)                    # (T + 1, 6, 6)
            d0 = torch.matmul(resp.reshape(T + 1, 2 * m, 6), J.transpose(1, 2).contiguous())
            y0.append(torch.cat([rel[:T, arm].detach(), d0.reshape(T + 1, -1)[:T]], 1))
        y = dopri5(f, torch.cat(y0), ts[:T].repeat(2), 0.0, **tol)[0]
        return [[a[:, :6], a[:, 6:].reshape(T, m, 12)] for a in (y[:T], y[T:])]


class Gradient:
    """Loss and gradient of the live-subhalo stream through the discrete adjoint: forward with
    checkpoints (or every row kept), then the whole reverse chain."""

    @staticmethod
    def draw(rng):
        return dict(steps=log_int(rng, 300, 4000), per_step=log_int(rng, 1, 25),
                    sources=log_int(rng, 5, 64), checkpoint=rng.choice([1, 50, 100, 100]))

    @staticmethod
    def prepare(case, seed):
        from streamsculptor_amd.adjoint import StreamModel
        w0, sub, m, rs, ts = Live.inputs(case, seed)
        model = StreamModel(ts, sub, rs, W.MSAT, case["per_step"], seed=seed % 1000,
                            checkpoint_every=case["checkpoint"])
        g = torch.Generator(device="cuda").manual_seed(seed)
        n = case["steps"] * case["per_step"]
        # a target stream: points along the progenitor's recent orbit, a stream's width apart
        rows = back_rows(HOST, jitter(W.PROG_TODAY, seed), -1.0, 60)[:, :3]
        at = torch.randint(0, 61, (n,), generator=g, device="cuda")
        target = gpu(rows)[at] + 0.2 * torch.randn(n, 3, generator=g, dtype=F64, device="cuda")
        return dict(model=model, target=target, m=m, w0=w0,
                    halo=np.array([W.HOST["m_halo"], W.HOST["rs_halo"]]))

    @staticmethod
    def run(s):
        from streamsculptor_amd.adjoint import stream_loss
        halo, m, w0 = (gpu(s[k]).requires_grad_(True) for k in ("halo", "m", "w0"))
        loss = stream_loss(halo, m, w0, s["model"], s["target"])
        loss.backward()
        return dict(loss=loss.detach(), halo=halo.grad, m=m.grad, w0=w0.grad)

    @staticmethod
    def work(case):
        # forward, re-run and reverse sweep: gradient twice, Hessian-vector product and the
        # source adjoints once
        per = (2 * flops.plain(case["sources"]) + flops.HOST_HESSIAN + 40
               + 40 * case["sources"])
        return dict(bytes=case["steps"] * case["per_step"] * 120.0
                    + 48.0 * (case["steps"] + 1) * case["sources"],
                    flops=float(W.particle_steps(case["per_step"], case["steps"])) * per)

    @staticmethod
    def exact(case, seed):
        if case["steps"] ** 2 * case["per_step"] * case["sources"] > 6e7:
            return None
        w0, sub, m, rs, _ = Live.inputs(case, seed)
        T, rs = case["steps"], gpu(rs)
        s = Gradient.prepare(case, seed)
        halo, ms, pw = (gpu(a).requires_grad_(True) for a in (s["halo"], m, w0))
        comps = HOST[:2] + [(NFW, [G * halo[0], halo[1]])]
        host = lambda x, k: -host_terms(comps, x)[1]  # noqa: E731
        track = leapfrog(host, gpu(sub), None, W.DT, T, keep=True)[..., :3]
        full = lambda x, k: host(x, k) - plummer_terms(x, track[k], G * ms, rs)[1]  # noqa: E731
        prog = leapfrog(full, pw[None], None, W.DT, T, keep=True)[:T, 0]
        rows, start = spray_rows(prog, host_terms(comps, prog[:, :3], True)[2], W.MSAT,
                                 case["per_step"], seed % 1000)
        out = leapfrog(full, rows, start, W.DT, T)
        loss = ((out[:, :3] - s["target"]) ** 2).sum()
        g = torch.autograd.grad(loss, [halo, ms, pw])
        return dict(loss=loss.detach(), halo=g[0], m=g[1], w0=g[2])


# parameter shapes of the 3-256-256-256-4 network, in the order of its parameter vector
SHAPES = [(256, 3), (256,), (256, 256), (256,), (256, 256), (256,), (4, 256), (4,)]


def split(p):
    out, o = [], 0
    for s in SHAPES:
        n = int(np.prod(s))
        out.append(p[o:o + n].reshape(s))
        o += n
    return out


def network(p, x, hidden=False):
    """The network in the parameters' own precision."""
    w1, b1, w2, b2, w3, b3, w4, b4 = split(p)
    for w, b in ((w1, b1), (w2, b2), (w3, b3)):
        x = torch.nn.functional.silu(x @ w.T + b)
    return x if hidden else x @ w4.T + b4


class Train:
    """One training iteration of the clump-force network: forward, weighted loss, gradients and
    the Adam step on a minibatch."""
    HALF = 25.0

    @staticmethod
    def draw(rng):
        return dict(batch=log_int(rng, 500, 32768))

    @staticmethod
    def inputs(case, seed):
        """(x, target, weight) of clump-force labels, and an optimiser state under way."""
        from streamsculptor_amd.mlp import init_params
        pos, m, rs = W.clump_table(seed=seed)
        xyz = gpu(orbits(case["batch"], seed)[:, :3])
        phi, g, _ = plummer_chunked(xyz, gpu(pos), gpu(G * m), gpu(rs))
        size = g.norm(dim=1)
        target = torch.cat([(phi / phi.std())[:, None], g / size.square().mean().sqrt()], 1)
        weight = 1.0 / (1.0 + (size / (30.0 * size.median())) ** 2)
        p = torch.as_tensor(init_params(seed % 1000), device="cuda")
        r = torch.Generator(device="cuda").manual_seed(seed)
        mom = 1e-3 * torch.randn(p.shape, generator=r, device="cuda")
        var = 1e-6 * (0.5 + torch.rand(p.shape, generator=r, device="cuda"))
        return (xyz / Train.HALF).float(), target.float(), weight.float(), p, mom, var

    @staticmethod
    def prepare(case, seed):
        from streamsculptor_amd.mlp import MLP
        x, t, w, p, mom, var = Train.inputs(case, seed)
        net = MLP(params=p)
        net.m.copy_(mom)
        net.v.copy_(var)
        net.step = 2000
        return dict(net=net, x=x, t=t, w=w)

    @staticmethod
    def run(s):
        net = s["net"]
        loss, y = net.loss_backward(s["x"], s["t"], s["w"])
        net.adam(1e-3)
        return dict(loss=loss, y=y, grads=net.grads, params=net.params, m=net.m, v=net.v)

    @staticmethod
    def work(case):
        return dict(bytes=case["batch"] * 48.0 + 4.0 * 133636 * 8,
                    flops=3.0 * flops.mlp() * case["batch"])

    @staticmethod
    def exact(case, seed):
        x, t, w, p, mom, var = (a.double() for a in Train.inputs(case, seed))
        p.requires_grad_(True)
        y = network(p, x)
        loss = (w[:, None] * (y - t) ** 2).sum() / w.sum()
        g = torch.autograd.grad(loss, p)[0]
        mom, var = 0.9 * mom + 0.1 * g, 0.999 * var + 0.001 * g * g
        new = p.detach() - 1e-3 * (mom / (1 - 0.9 ** 2001)) / (
            torch.sqrt(var / (1 - 0.999 ** 2001)) + 1e-8)
        return dict(loss=loss.detach().reshape(1), y=y.detach(), grads=g, params=new, m=mom, v=var)


class Surrogate:
    """Orbits through the learned clump force with the exact sum in flagged cells: forward, or
    forward and adjoint."""
    HALF, CELLS = 25.0, 64

    @staticmethod
    def draw(rng):
        return dict(n=log_int(rng, 500, 60000), steps=rng.randint(20, 100),
                    sources=log_int(rng, 64, 512), gradient=rng.random() < 0.5)

    @staticmethod
    def model(case, seed):
        """Network parameters and scaling of a fit to the clumps, and the flagged cells."""
        from streamsculptor_amd.mlp import init_params
        pos, m, rs = W.clump_table(n=case["sources"], seed=seed)
        xyz = orbits(4096, seed + 1)[:, :3]
        d = xyz[:, None] - pos
        s2 = (d * d).sum(-1) + rs * rs
        phi, g = -(G * m / np.sqrt(s2)).sum(1), ((G * m * s2 ** -1.5)[..., None] * d).sum(1)
        ps, gs = float(phi.std()), float(np.sqrt((g * g).sum(1).mean()))
        p = torch.as_tensor(init_params(seed % 1000))
        feat = network(p.double(), torch.as_tensor(xyz / Surrogate.HALF), hidden=True).numpy()
        feat = np.hstack([feat, np.ones((4096, 1))])
        lab = np.hstack([phi[:, None] / ps, g / gs])
        sol = np.linalg.solve(feat.T @ feat + 1e-3 * np.eye(257), feat.T @ lab)
        parts = [a.clone() for a in split(p)]
        parts[6], parts[7] = torch.as_tensor(sol[:256].T.copy()), torch.as_tensor(sol[256].copy())
        p = torch.cat([a.reshape(-1).float() for a in parts])
        n, cell = Surrogate.CELLS, 2.0 * Surrogate.HALF / Surrogate.CELLS
        # the cells nearest to a clump take the exact sum: 4 % of those orbits visit
        ax = gpu((np.arange(n) + 0.5) * cell - Surrogate.HALF)
        mid = torch.stack(torch.meshgrid(ax, ax, ax, indexing="ij"), -1).reshape(-1, 3)
        near = torch.cat([((c[:, None] - gpu(pos)) ** 2).sum(-1).min(1).values
                          for c in mid.split(1 << 15)])
        r = mid.norm(dim=1)
        lim = torch.quantile(near[(r > 7) & (r < 20)], 0.04)
        return pos, m, rs, p, ps, gs, (near < lim).reshape(n, n, n).to(torch.uint8), cell

    @staticmethod
    def inputs(case, seed):
        g = torch.Generator(device="cuda").manual_seed(seed)
        start = np.sort(np.random.default_rng(seed).integers(0, case["steps"] // 2, case["n"]))
        return (gpu(orbits(case["n"], seed)), start.astype(np.int32),
                torch.randn(case["n"], 6, generator=g, dtype=F64, device="cuda"))

    @staticmethod
    def prepare(case, seed):
        from streamsculptor_amd.main import usys
        from streamsculptor_amd.mlp import MLP
        from streamsculptor_amd.potential import PlummerClumps
        from streamsculptor_amd.surrogate import ClumpSurrogate, Scaling
        pos, m, rs, p, ps, gs, flags, cell = Surrogate.model(case, seed)
        half = Surrogate.HALF
        sur = ClumpSurrogate(W.host_potential(), PlummerClumps(m, rs, pos, units=usys), MLP(params=p),
                             Scaling((0.0,) * 3, (half,) * 3, ps, gs), flags, (-half,) * 3,
                             (cell,) * 3, (Surrogate.CELLS,) * 3)
        w0, start, lam = Surrogate.inputs(case, seed)
        return dict(sur=sur, w0=w0, start=torch.as_tensor(start, device="cuda"), lam=lam, case=case)

    @staticmethod
    def run(s):
        T = s["case"]["steps"]
        if not s["case"]["gradient"]:
            out, count = s["sur"].leapfrog(s["w0"], 0.0, W.DT, T, start=s["start"])
            return dict(w=out, fallback=count)
        adj = s["sur"].adjoint(s["w0"], 0.0, W.DT, T, start=s["start"])
        out = adj.forward()
        back = adj.backward(s["lam"])
        return dict(w=out, lam0=back["lam0"], g_host=back["g_host"], fallback=back["fallback"])

    @staticmethod
    def work(case):
        rows = case["n"] * case["steps"] * 0.75
        return dict(bytes=case["n"] * 96.0 * (2 if case["gradient"] else 1) + 4.0 * 133636,
                    flops=rows * (flops.mlp() + (flops.mlp_input_vjp() if case["gradient"] else 0)))

    @staticmethod
    def exact(case, seed):
        pos, m, rs, p, _, gs, flags, cell = Surrogate.model(case, seed)
        pos, gm, rs, p, half = gpu(pos), gpu(G * m), gpu(rs), p.double().cuda(), Surrogate.HALF
        w0, start, lam = Surrogate.inputs(case, seed)
        start, T, dt = torch.as_tensor(start, device="cuda"), case["steps"], W.DT
        par = torch.tensor([[q[0], q[1]] for _, q in HOST], dtype=F64, device="cuda",
                           requires_grad=True)
        comps = [(k, [par[i, 0], par[i, 1], *q[2:]]) for i, (k, q) in enumerate(HOST)]

        def acc(x, k):
            ijk = torch.floor((x.detach() + half) / cell).long()
            inside = ((ijk >= 0) & (ijk < Surrogate.CELLS)).all(1)
            i = ijk.clamp(0, Surrogate.CELLS - 1)
            exact_sum = ~inside | (flags[i[:, 0], i[:, 1], i[:, 2]] != 0)
            g = gs * network(p, x / half)[:, 1:]
            rows = torch.nonzero(exact_sum).flatten()
            if rows.numel():
                g = g.index_put((rows,), plummer_terms(x[rows], pos, gm, rs)[1])
            return -host_terms(comps, x)[1] - g

        with torch.no_grad():
            rows = leapfrog(acc, w0, start, dt, T, keep=True)
        if not case["gradient"]:
            return dict(w=rows[-1], fallback=None)
        lx, lv = lam[:, :3], lam[:, 3:]
        gpar = torch.zeros_like(par)
        for k in range(T, -1, -1):
            on, first = (start <= k)[:, None], (start == k)[:, None]
            if k < T:
                lh = torch.where(on, lv + dt * lx, lv)
                wk = torch.where(on, torch.where(first, 0.5 * dt * lh, dt * lh), 0.0)
                lv = lh
            else:
                wk = 0.5 * dt * lv
            x = rows[k][:, :3].detach().requires_grad_(True)
            gx, gp = torch.autograd.grad((acc(x, k) * wk).sum(), [x, par])
            lx, gpar = lx + gx, gpar + gp
        return dict(w=rows[-1], lam0=torch.cat([lx, lv], 1), g_host=gpar, fallback=None)


PATHS = dict(orbit=Orbit, evaluate=Evaluate, stream=Stream, batch=Batch, live=Live, clumps=Clumps,
             responses=Responses, derivs=Derivs, gradient=Gradient, train=Train,
             surrogate=Surrogate)


# ---------------------------------------------------------------------------------------------
def listed():
    return [
        # one adaptive orbit with saved rows: the call a user makes most, latency only
        dict(name="orbit", path="orbit", n=1, age=2500, saves=251, solver="dopri5",
             potential="milky way"),
        # labels and tidal fields at many points of the clumpy halo
        dict(name="evaluate", path="evaluate", n=262144, sources=512),
        # the plain fixed-step stream, 8000 particles
        dict(name="stream", path="stream", steps=4000, solver="leapfrog", potential="host"),
        # the adaptive stream in the Milky Way model, the stream generators' default solver
        dict(name="stream-adaptive", path="stream", steps=2000, solver="dopri5",
             potential="milky way"),
        # a full batch of perturbed GD-1-like streams
        dict(name="batch", path="batch", sims=700, strip=2000),
        # 1e5 particles in 64 live subhalos
        dict(name="live", path="live", steps=4000, per_step=25, sources=64),
        # 4e5 particles in 512 clumps: the largest direct sum
        dict(name="clumps", path="clumps", steps=4000, per_step=100, sources=512),
        # 8e4 particles with 64 response vectors each
        dict(name="responses", path="responses", steps=4000, per_step=20, sources=64,
             radius=False),
        # adaptive mass and radius responses to 128 Hernquist subhalos
        dict(name="derivs", path="derivs", steps=1000, sources=128, profile="hernquist"),
        # loss and gradient of the live-subhalo stream, checkpoints every 100 steps
        dict(name="gradient", path="gradient", steps=4000, per_step=25, sources=64,
             checkpoint=100),
        # a training iteration at the default minibatch
        dict(name="train", path="train", batch=8192),
        # the learned force forward and through its adjoint
        dict(name="surrogate", path="surrogate", n=60000, steps=100, sources=512, gradient=True),
    ]


def draw(rng):
    path = rng.choice(sorted(PATHS))
    return dict(path=path, **PATHS[path].draw(rng))


def prepare(case, seed):
    return PATHS[case["path"]], PATHS[case["path"]].prepare(case, int(seed))


def run(state):
    path, s = state
    return path.run(s)


def work(case):
    return PATHS[case["path"]].work(case)


def exact(case, seed):
    return PATHS[case["path"]].exact(case, int(seed))
