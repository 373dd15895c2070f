// First-order perturbation responses (the fields-interface OTF perturbation ODE) on gfx950.
//
// Per particle the state is the unperturbed row w = (x, v) in the host potential plus, for
// every perturbing source j (Plummer spheres, or Hernquist spheres for straight-line Hernquist
// subhalos), the response dw_j = d w / d eps_j at eps = 0 (mass block)
// and optionally d^2 w / d a_j d eps_j (radius block).  Discretisation: the exact derivative of
// the kick-drift-kick map of Phi_host + sum_j eps_j Phi_j, i.e. the responses follow
//   d(dx)/dt = dv,  d(dv)/dt = -grad Phi_j(x) - H(x) dx          (mass)
//   d(rx)/dt = rv,  d(rv)/dt = -grad(dPhi_j/da_j)(x) - H(x) rx    (radius)
// as in reference MassRadiusPerturbation_OTF.term (streamsculptor/fields.py:175-206), with
// dPhi_j/da_j the structural potential of SubhaloLinePotential_dRadius (potential.py:852-904)
// or SubhaloLinePotentialCustom_dRadius_fromFunc (potential.py:1215-1268).
//
// Layout: L = ceil(m / G) lanes per particle; lane g of a particle owns the G responses g,
// g + L, g + 2L, ... (strided: at every response slot the L lanes read consecutive source
// records, which keeps their LDS reads free of bank conflicts).  With a workspace the
// grid is cut into segments of rows: base_rows (one particle per lane) advances the base orbits
// through a segment and records, at every row a particle is kicked at, its position and the host
// Hessian; response_rows then advances the responses through the segment from those records.
// One launch carries the base rows of segment s + 1 beside the responses of segment s: the first
// waits for memory (72 B a particle and row), the second for FP64 issue (a grid of fewer than two
// segments of 64 rows has one, its responses after its base rows).  Without a workspace
// perturb_kernel has each of the L lanes recompute the base orbit and the host Hessian (2.2x the
// arithmetic of the split form, measured by counters).
// Velocities are carried at half steps so that forces are consumed as soon as they are formed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <string>

#include "ssc_device.h"
#include "ssc_sources_lds.h"

namespace ssc {

constexpr int PT_BLOCK = 256;

// host gradient and Hessian (upper triangle filled into all 9) at one point
template <int HS>
__device__ __forceinline__ void host_grad_hess(const ssc_host_potential& hp, double x, double y,
                                               double z, double* g, double* H) {
  double phi;
  host_full_sig<HS, true>(hp, x, y, z, phi, g, H);
}

// The same from the components' four numbers, accumulated into g and H's upper triangle: the
// spherical components are added up before their 3 x 3 terms are formed.
template <int HS>
__device__ __forceinline__ void host_quads(const ssc_host_potential& hp, double x, double y,
                                           double z, double* g, double* H) {
  if constexpr (HS == HS_GENERIC) {
    for (int c = 0; c < hp.n_components; ++c) quad_add(comp_quad(hp.c[c], x, y, z), x, y, g, H);
  } else {
    const CompQuad d = comp_quad<hs_kind(HS, 0)>(hp.c[0], x, y, z);
    CompQuad q = comp_quad<hs_kind(HS, 1)>(hp.c[1], x, y, z);
    const CompQuad q2 = comp_quad<hs_kind(HS, 2)>(hp.c[2], x, y, z);
    q.f += q2.f;
    q.k += q2.k;
    if constexpr (hs_components(HS) > 3) {
      const CompQuad q3 = comp_quad<hs_kind(HS, 3)>(hp.c[3], x, y, z);
      q.f += q3.f;
      q.k += q3.k;
    }
    quad_add(d, x, y, g, H);
    quad_add(q, x, y, g, H);
  }
}

template <int SK, int G, int RAD, int HS>
__global__ __launch_bounds__(PT_BLOCK) void perturb_kernel(
    ssc_host_potential hp, ssc_sources pert, const double* __restrict__ w0,
    const double* __restrict__ dw0, const int32_t* __restrict__ start, int64_t n, int m, int L,
    double t0, double dt, int nsteps, double* __restrict__ w_out, double* __restrict__ dw_out) {
  extern __shared__ __align__(16) char lds_raw[];
  __shared__ int kmin_sh;
  constexpr int DD = RAD ? 12 : 6;
  constexpr bool HQ = SK == SSC_SRC_LINE_HERNQUIST;
  const int ppb = PT_BLOCK / L;
  const int lp = threadIdx.x / L, grp = threadIdx.x - lp * L;
  const int64_t i = (int64_t)blockIdx.x * ppb + lp;
  const bool valid = lp < ppb && i < n;

  double x = 1.0, y = 0.0, z = 0.0, vx = 0.0, vy = 0.0, vz = 0.0;
  double dx[G][3], dv[G][3], rx[RAD ? G : 1][3], rv[RAD ? G : 1][3];
  int s = nsteps;
  if (valid) {
    const double* w = w0 + 6 * i;
    x = w[0]; y = w[1]; z = w[2]; vx = w[3]; vy = w[4]; vz = w[5];
    s = start ? start[i] : 0;
    s = s < 0 ? 0 : (s > nsteps ? nsteps : s);
  }
#pragma unroll
  for (int q = 0; q < G; ++q) {
    const int j = grp + L * q;
    const bool ok = valid && j < m && dw0;
    const double* d = ok ? dw0 + ((int64_t)i * m + j) * DD : nullptr;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      dx[q][c] = ok ? d[c] : 0.0;
      dv[q][c] = ok ? d[3 + c] : 0.0;
      if (RAD) {
        rx[q][c] = ok ? d[6 + c] : 0.0;
        rv[q][c] = ok ? d[9 + c] : 0.0;
      }
    }
  }
  if (threadIdx.x == 0) kmin_sh = INT_MAX;
  __syncthreads();
  atomicMin(&kmin_sh, s);
  SourceLDS<SK> lds;
  lds.init(pert, lds_raw);
  __syncthreads();
  const int kmin = kmin_sh;
  const double h = 0.5 * dt;

  // Forces at grid row k: base acceleration a, and for every owned response the force
  // F = -grad Phi_j - H dx (and the radius-block force), applied as vel += c * F.
  auto apply = [&](int k, double c, bool move) {
    const double t = t0 + k * dt;
    double g[3], H[9];
    host_grad_hess<HS>(hp, x, y, z, g, H);
    if (move) {
      vx -= c * g[0]; vy -= c * g[1]; vz -= c * g[2];
    }
#pragma unroll
    for (int q = 0; q < G; ++q) {
      const int j = grp + L * q;
      double sx, sy, sz, gm, q2;
      const bool act = (j < m) && lds.get(k, t, j, sx, sy, sz, gm, q2);
      double fx = 0.0, fy = 0.0, fz = 0.0, ux = 0.0, uy = 0.0, uz = 0.0;
      if (act) {
        const double ex = x - sx, ey = y - sy, ez = z - sz;
        if (HQ) {  // Hernquist (q2 holds a): f = G m / (r (r + a)^2)
          const double r2 = fma(ex, ex, fma(ey, ey, ez * ez));
          const double ir = rsq(r2);
          const double ia = 1.0 / fma(r2, ir, q2);
          const double f = gm * ir * ia * ia;
          fx = f * ex; fy = f * ey; fz = f * ez;
          if (RAD) {  // grad of dPhi_j/da_j = -2 G m e / (r (r + a)^3)
            const double r5 = -2.0 * f * ia;
            ux = r5 * ex; uy = r5 * ey; uz = r5 * ez;
          }
        } else {  // Plummer (q2 holds a^2)
          const double s2 = fma(ex, ex, fma(ey, ey, fma(ez, ez, q2)));
          const double is = rsq(s2);
          const double f = gm * is * is * is;
          fx = f * ex; fy = f * ey; fz = f * ez;
          if (RAD) {  // grad of dPhi_j/da_j = -3 G m a e / s^5
            const double r5 = -3.0 * f * sqrt(q2) * is * is;
            ux = r5 * ex; uy = r5 * ey; uz = r5 * ez;
          }
        }
      }
      if (move) {
        const double hx = H[0] * dx[q][0] + H[1] * dx[q][1] + H[2] * dx[q][2];
        const double hy = H[3] * dx[q][0] + H[4] * dx[q][1] + H[5] * dx[q][2];
        const double hz = H[6] * dx[q][0] + H[7] * dx[q][1] + H[8] * dx[q][2];
        dv[q][0] -= c * (fx + hx);
        dv[q][1] -= c * (fy + hy);
        dv[q][2] -= c * (fz + hz);
        if (RAD) {
          const double px = H[0] * rx[q][0] + H[1] * rx[q][1] + H[2] * rx[q][2];
          const double py = H[3] * rx[q][0] + H[4] * rx[q][1] + H[5] * rx[q][2];
          const double pz = H[6] * rx[q][0] + H[7] * rx[q][1] + H[8] * rx[q][2];
          rv[q][0] -= c * (ux + px);
          rv[q][1] -= c * (uy + py);
          rv[q][2] -= c * (uz + pz);
        }
      }
    }
  };

  if (kmin < nsteps) {
    lds.stage(pert, kmin, nsteps + 1);
    apply(kmin, h, valid && s == kmin);  // first half kick of particles starting at kmin
  }
  for (int k = kmin; k < nsteps; ++k) {
    lds.stage(pert, k, nsteps + 1);
    const bool act = valid && k >= s;
    if (act) {
      x += dt * vx; y += dt * vy; z += dt * vz;
#pragma unroll
      for (int q = 0; q < G; ++q) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          dx[q][c] += dt * dv[q][c];
          if (RAD) rx[q][c] += dt * rv[q][c];
        }
      }
    }
    // active: full kick to the next half step (or the closing half kick at the last row);
    // starting at k + 1: its opening half kick
    const bool last = (k + 1 == nsteps);
    const bool starts = valid && s == k + 1 && s < nsteps;
    apply(k + 1, (act && !last) ? dt : h, act || starts);
  }
  if (valid) {
    if (grp == 0) {
      double* o = w_out + 6 * i;
      o[0] = x; o[1] = y; o[2] = z; o[3] = vx; o[4] = vy; o[5] = vz;
    }
#pragma unroll
    for (int q = 0; q < G; ++q) {
      const int j = grp + L * q;
      if (j < m) {
        double* o = dw_out + ((int64_t)i * m + j) * DD;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          o[c] = dx[q][c];
          o[3 + c] = dv[q][c];
          if (RAD) {
            o[6 + c] = rx[q][c];
            o[9 + c] = rv[q][c];
          }
        }
      }
    }
  }
}

// ------------------------------------------------------------------------------------------
// Split form.  The kick rows of a particle starting at s < nsteps are s (opening half kick),
// s + 1 .. nsteps - 1 (a drift, then a full kick) and nsteps (a drift, then the closing half
// kick) -- the steps perturb_kernel takes.  A segment covers rows [ka, kb].  Record of row k:
// base position and the upper triangle of the host Hessian, [kb - ka + 1][n][9].
// ------------------------------------------------------------------------------------------
constexpr int PR_REC = 9;

__global__ void pt_zero_kernel(double* __restrict__ p, int64_t n) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n) p[e] = 0.0;
}

// Base orbits in place in w (initialised to w0), rows [ka, kb]: one particle per lane.  A wave's
// 64 records of a row go through LDS, so that they leave as nine stores of 512 consecutive bytes
// (80,000 orbits x 4,000 rows 6.3 ms by itself; 7.6 ms written by their own lanes 72 B apart), while
// there are enough waves for that to be a matter of bandwidth: below 32,768 orbits a row's way
// through LDS is a part of its chain, and the lanes write their own (60 rows, 50 orbits x 64 sources
// 0.087 ms against 0.104, 20,000 x 64 0.165 against 0.171).
constexpr int BASE_LDS = PT_BLOCK * PR_REC * 8;
constexpr int64_t BASE_DIRECT = 32768;

template <int HS>
__device__ __forceinline__ void base_rows(const ssc_host_potential& hp, int block, char* lds_raw,
                                          double* __restrict__ w, const int32_t* __restrict__ start,
                                          int64_t n, double dt, int nsteps, int ka, int kb,
                                          double* __restrict__ rows) {
  const int lane = threadIdx.x & 63;
  const int64_t i0 = (int64_t)block * PT_BLOCK + (threadIdx.x & ~63);  // the wave's first particle
  const int64_t i = i0 + lane;
  if (i0 >= n) return;  // whole waves only: the others keep together below
  int s = i < n ? (start ? start[i] : 0) : nsteps;
  s = s < 0 ? 0 : (s > nsteps ? nsteps : s);
  const bool moves = i < n && s < nsteps && s <= kb;
  double* wi = w + 6 * i;
  double x = 1.0, y = 0.0, z = 0.0, vx = 0.0, vy = 0.0, vz = 0.0;
  if (moves) {
    x = wi[0]; y = wi[1]; z = wi[2]; vx = wi[3]; vy = wi[4]; vz = wi[5];
  }
  int first = moves ? (ka > s ? ka : s) : INT_MAX;  // the wave's first row
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) first = min(first, __shfl_xor(first, o, 64));
  const double h = 0.5 * dt;
  double* buf = reinterpret_cast<double*>(lds_raw) + (threadIdx.x >> 6) * (64 * PR_REC);
  const int64_t tail = (n - i0) * PR_REC;  // doubles of the wave's particles that exist
  for (int k = first; k <= kb; ++k) {
    const bool on = moves && k >= s;
    if (on && k > s) {
      x += dt * vx; y += dt * vy; z += dt * vz;
    }
    double g[3] = {0.0, 0.0, 0.0}, H[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) H[q] = 0.0;
    host_quads<HS>(hp, x, y, z, g, H);
    // records of particles that have not started are written and never read
    if (n < BASE_DIRECT) {
      if (i < n) {
        double* r = rows + ((int64_t)(k - ka) * n + i) * PR_REC;
        r[0] = x; r[1] = y; r[2] = z;
        r[3] = H[0]; r[4] = H[1]; r[5] = H[2]; r[6] = H[4]; r[7] = H[5]; r[8] = H[8];
      }
    } else {
      double* b = buf + lane * PR_REC;
      b[0] = x; b[1] = y; b[2] = z;
      b[3] = H[0]; b[4] = H[1]; b[5] = H[2]; b[6] = H[4]; b[7] = H[5]; b[8] = H[8];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      double* r = rows + ((int64_t)(k - ka) * n + i0) * PR_REC;
#pragma unroll
      for (int e = 0; e < PR_REC; ++e) {
        const int o = 64 * e + lane;
        if (o < tail) r[o] = buf[o];
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (on) {
      const double c = (k == s || k == nsteps) ? h : dt;
      vx -= c * g[0]; vy -= c * g[1]; vz -= c * g[2];
    }
  }
  if (moves) {
    wi[0] = x; wi[1] = y; wi[2] = z; wi[3] = vx; wi[4] = vy; wi[5] = vz;
  }
}

// Responses in place in dw ([n][m][DD], initialised to dw0 or zeros) through rows [ka, kb].
template <int SK, int G, int RAD>
__device__ __forceinline__ void response_rows(const ssc_sources& pert, int block, char* lds_raw,
                                              int& kmin_sh, const double* __restrict__ rows,
                                              const int32_t* __restrict__ start, int64_t n, int m,
                                              int L, double t0, double dt, int nsteps, int ka,
                                              int kb, double* __restrict__ dw) {
  constexpr int DD = RAD ? 12 : 6;
  constexpr bool HQ = SK == SSC_SRC_LINE_HERNQUIST;
  constexpr bool FOLD = (SK == SSC_SRC_STATIC || SK == SSC_SRC_TRACK) && !RAD;
  const int ppb = PT_BLOCK / L;
  const int lp = threadIdx.x / L, grp = threadIdx.x - lp * L;
  const int64_t i = (int64_t)block * ppb + lp;
  const bool valid = lp < ppb && i < n;
  int s = nsteps;
  if (valid) {
    s = start ? start[i] : 0;
    s = s < 0 ? 0 : (s > nsteps ? nsteps : s);
  }
  const bool moves = valid && s < nsteps && s <= kb;
  double dx[G][3], dv[G][3], rx[RAD ? G : 1][3], rv[RAD ? G : 1][3];
#pragma unroll
  for (int q = 0; q < G; ++q) {
    const int j = grp + L * q;
    const bool ok = moves && j < m;
    const double* d = ok ? dw + ((int64_t)i * m + j) * DD : nullptr;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      dx[q][c] = ok ? d[c] : 0.0;
      dv[q][c] = ok ? d[3 + c] : 0.0;
      if (RAD) {
        rx[q][c] = ok ? d[6 + c] : 0.0;
        rv[q][c] = ok ? d[9 + c] : 0.0;
      }
    }
  }
  if (threadIdx.x == 0) kmin_sh = INT_MAX;
  __syncthreads();
  if (moves) atomicMin(&kmin_sh, s);
  SourceLDS<SK> lds;
  lds.init(pert, lds_raw);
  __syncthreads();
  const int kfirst = kmin_sh < ka ? ka : kmin_sh;  // block-uniform
  const double h = 0.5 * dt;
  for (int k = kfirst; k <= kb; ++k) {
    lds.stage(pert, k, nsteps + 1);
    if (!(moves && k >= s)) continue;
    const double* r = rows + ((int64_t)(k - ka) * n + i) * PR_REC;
    const double x = r[0], y = r[1], z = r[2];
    const double H[9] = {r[3], r[4], r[5], r[4], r[6], r[7], r[5], r[7], r[8]};
    if (k > s) {
#pragma unroll
      for (int q = 0; q < G; ++q)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          dx[q][c] += dt * dv[q][c];
          if (RAD) rx[q][c] += dt * rv[q][c];
        }
    }
    const double t = t0 + k * dt;
    const double c = (k == s || k == nsteps) ? h : dt;
    if constexpr (FOLD) {
      // Plummer sources that are always active: no branch per response, the folded
      // reciprocal-square-root correction of plummer_grad_k, and the kick c folded into the
      // Hessian (once a row) and the source's factor, so that a velocity component takes four
      // FMAs: 28 instructions a response.  A slot beyond the last source computes a response
      // that is never stored.
      const double C[6] = {-c * H[0], -c * H[1], -c * H[2], -c * H[4], -c * H[5], -c * H[8]};
#pragma unroll
      for (int q = 0; q < G; ++q) {
        const int j = grp + L * q;
        double sx, sy, sz, q2, c1, c2;
        lds.get_k(k, j < m ? j : m - 1, sx, sy, sz, q2, c1, c2);
        const double ex = x - sx, ey = y - sy, ez = z - sz;
        const double s2 = fma(ex, ex, fma(ey, ey, fma(ez, ez, q2)));
        const double yr = __builtin_amdgcn_rsq(s2);
        const double y2 = yr * yr;
        const double f = (-c * yr) * y2 * fma(s2 * y2, c1, c2);
        double* u = dx[q];
        dv[q][0] = fma(f, ex, fma(C[2], u[2], fma(C[1], u[1], fma(C[0], u[0], dv[q][0]))));
        dv[q][1] = fma(f, ey, fma(C[4], u[2], fma(C[3], u[1], fma(C[1], u[0], dv[q][1]))));
        dv[q][2] = fma(f, ez, fma(C[5], u[2], fma(C[4], u[1], fma(C[2], u[0], dv[q][2]))));
      }
      continue;
    }
#pragma unroll
    for (int q = 0; q < G; ++q) {
      const int j = grp + L * q;
      double sx, sy, sz, gm, q2;
      const bool act = (j < m) && lds.get(k, t, j, sx, sy, sz, gm, q2);
      double fx = 0.0, fy = 0.0, fz = 0.0, ux = 0.0, uy = 0.0, uz = 0.0;
      if (act) {
        const double ex = x - sx, ey = y - sy, ez = z - sz;
        if (HQ) {  // Hernquist (q2 holds a): f = G m / (r (r + a)^2)
          const double r2 = fma(ex, ex, fma(ey, ey, ez * ez));
          const double ir = rsq(r2);
          const double ia = 1.0 / fma(r2, ir, q2);
          const double f = gm * ir * ia * ia;
          fx = f * ex; fy = f * ey; fz = f * ez;
          if (RAD) {  // grad of dPhi_j/da_j = -2 G m e / (r (r + a)^3)
            const double r5 = -2.0 * f * ia;
            ux = r5 * ex; uy = r5 * ey; uz = r5 * ez;
          }
        } else {  // Plummer (q2 holds a^2)
          const double s2 = fma(ex, ex, fma(ey, ey, fma(ez, ez, q2)));
          const double is = rsq(s2);
          const double f = gm * is * is * is;
          fx = f * ex; fy = f * ey; fz = f * ez;
          if (RAD) {  // grad of dPhi_j/da_j = -3 G m a e / s^5
            const double r5 = -3.0 * f * sqrt(q2) * is * is;
            ux = r5 * ex; uy = r5 * ey; uz = r5 * ez;
          }
        }
      }
      const double hx = H[0] * dx[q][0] + H[1] * dx[q][1] + H[2] * dx[q][2];
      const double hy = H[3] * dx[q][0] + H[4] * dx[q][1] + H[5] * dx[q][2];
      const double hz = H[6] * dx[q][0] + H[7] * dx[q][1] + H[8] * dx[q][2];
      dv[q][0] -= c * (fx + hx);
      dv[q][1] -= c * (fy + hy);
      dv[q][2] -= c * (fz + hz);
      if (RAD) {
        const double px = H[0] * rx[q][0] + H[1] * rx[q][1] + H[2] * rx[q][2];
        const double py = H[3] * rx[q][0] + H[4] * rx[q][1] + H[5] * rx[q][2];
        const double pz = H[6] * rx[q][0] + H[7] * rx[q][1] + H[8] * rx[q][2];
        rv[q][0] -= c * (ux + px);
        rv[q][1] -= c * (uy + py);
        rv[q][2] -= c * (uz + pz);
      }
    }
  }
  if (moves) {
#pragma unroll
    for (int q = 0; q < G; ++q) {
      const int j = grp + L * q;
      if (j < m) {
        double* o = dw + ((int64_t)i * m + j) * DD;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          o[c] = dx[q][c];
          o[3 + c] = dv[q][c];
          if (RAD) {
            o[6 + c] = rx[q][c];
            o[9 + c] = rv[q][c];
          }
        }
      }
    }
  }
}

// One launch: base rows [na, nb_] of the next segment in the first bblocks blocks, the responses
// of rows [ka, kb] in the others.
template <int SK, int G, int RAD, int HS>
__global__ __launch_bounds__(PT_BLOCK) void perturb_segment_kernel(
    ssc_host_potential hp, ssc_sources pert, int bblocks, double* __restrict__ w,
    const int32_t* __restrict__ start, int64_t n, int m, int L, double t0, double dt, int nsteps,
    int ka, int kb, const double* __restrict__ rows, int na, int nb_,
    double* __restrict__ next_rows, double* __restrict__ dw) {
  extern __shared__ __align__(16) char lds_raw[];
  __shared__ int kmin_sh;
  if ((int)blockIdx.x < bblocks)
    base_rows<HS>(hp, blockIdx.x, lds_raw, w, start, n, dt, nsteps, na, nb_, next_rows);
  else
    response_rows<SK, G, RAD>(pert, blockIdx.x - bblocks, lds_raw, kmin_sh, rows, start, n, m, L,
                              t0, dt, nsteps, ka, kb, dw);
}

// Responses per lane of the split form: two while the lanes of eight would give the chip fewer than
// two waves per SIMD, and with the radius block always (twelve numbers a response: 118 registers
// with two, 374 and one wave per SIMD with eight); eight otherwise, since a lane's row record and
// Hessian then serve eight responses.  Up to 512 sources with two (256 lanes a particle).
// Measured (ms, 2 / 4 / 8 a lane): 80,000 particles x 64 sources, 4,000 steps 26.1 / 22.8 / 21.0,
// with the radius block 40.0 / 40.5 / 54.3; 40,000 x 64, 2,000 steps 8.0 / 7.1 / 6.7; 8,100 x 33,
// 900 steps 2.00 / 2.08 / 2.33; 1,000 x 7, 500 steps 1.09 / 1.17 / 1.33.
static bool split_few(int64_t n, int m, bool radius) {
  if (m > 2 * PT_BLOCK) return false;
  int L = 1;
  while (8 * L < m) L <<= 1;
  return radius || n * L < (int64_t)2 * 1024 * 64;
}

// Rows of records to keep where there is room: two segments of an eighth of the grid each, so that
// all but an eighth of the base rows are formed beside responses, or all rows of a grid of fewer
// than two segments of 64.  Segments of an eighth and one of all rows (ms): 8,000 particles x 64
// sources, 4,000 steps 3.94 and 5.91 (0.6 and 2.3 GB), 1,000 x 7, 500 steps 0.51 and 0.68, 40,000 x
// 64, 1,000 steps 2.42 and 2.55; with fewer than 64 rows a segment the two parts' blocks no
// longer last each other out: 500,000 x 4, 100 steps 1.24 (13 rows) and 0.91.
static int64_t perturb_rows_wanted(int nsteps) {
  const int64_t r = std::max<int64_t>(64, ((int64_t)nsteps + 8) / 8);
  return 2 * r > nsteps ? (int64_t)nsteps + 1 : 2 * r;
}

// Rows of records that fit in workspace_bytes (0 when not even one does), no more than wanted.
static int64_t perturb_segment_rows(int64_t n, int nsteps, int64_t workspace_bytes) {
  return std::min(workspace_bytes / (n * PR_REC * 8), perturb_rows_wanted(nsteps));
}

// Segments take turns in the two halves of a workspace that holds at least two rows but not all.
static int64_t perturb_buffer_rows(int64_t E, int nsteps) {
  return E > nsteps || E < 2 ? E : E / 2;
}

template <int SK, int G, int RAD, int HS>
static int launch_perturb_split(const ssc_host_potential& hp, const ssc_sources& pert,
                                const double* w0, const double* dw0, const int32_t* start,
                                int64_t n, double t0, double dt, int nsteps, double* w_out,
                                double* dw_out, double* rows, int64_t E, hipStream_t st) {
  const int m = pert.n;
  constexpr int DD = RAD ? 12 : 6;
  int L = (m + G - 1) / G;
  int Lp = 1;
  while (Lp < L) Lp <<= 1;
  if (Lp > PT_BLOCK) return fail(SSC_E_LIMIT, "ssc_perturb_leapfrog: too many sources");
  const size_t lds = std::max<size_t>(SourceLDS<SK>::bytes(pert), BASE_LDS);
  if (lds > 60 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)perturb_segment_kernel<SK, G, RAD, HS>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return fail(SSC_E_HIP, std::string("hipFuncSetAttribute: ") + hipGetErrorString(e));
  }
  hipMemcpyAsync(w_out, w0, (size_t)n * 6 * 8, hipMemcpyDeviceToDevice, st);
  if (dw0)
    hipMemcpyAsync(dw_out, dw0, (size_t)n * m * DD * 8, hipMemcpyDeviceToDevice, st);
  else
    hipLaunchKernelGGL(pt_zero_kernel, dim3((unsigned)((n * m * DD + 255) / 256)), dim3(256), 0,
                       st, dw_out, n * m * DD);
  const unsigned bblocks = (unsigned)((n + PT_BLOCK - 1) / PT_BLOCK);
  const unsigned rblocks = (unsigned)((n + PT_BLOCK / Lp - 1) / (PT_BLOCK / Lp));
  const int64_t B = perturb_buffer_rows(E, nsteps);
  double* buf[2] = {rows, B < E ? rows + B * n * PR_REC : rows};
  auto launch = [&](unsigned nb, unsigned nr, int64_t ka, int64_t kb, const double* cur,
                    int64_t na, int64_t nbk, double* next) {
    hipLaunchKernelGGL((perturb_segment_kernel<SK, G, RAD, HS>), dim3(nb + nr), dim3(PT_BLOCK), lds,
                       st, hp, pert, (int)nb, w_out, start, n, m, Lp, t0, dt, nsteps, (int)ka,
                       (int)kb, cur, (int)na, (int)nbk, next, dw_out);
  };
  auto last = [&](int64_t ka) { return std::min<int64_t>(ka + B - 1, nsteps); };
  launch(bblocks, 0, 0, 0, buf[0], 0, last(0), buf[0]);
  int cur = 0;
  for (int64_t ka = 0; ka <= nsteps; ka += B) {
    const int64_t na = ka + B;
    const bool more = na <= nsteps;
    if (more && buf[0] != buf[1]) {
      launch(bblocks, rblocks, ka, last(ka), buf[cur], na, last(na), buf[cur ^ 1]);
      cur ^= 1;
    } else {
      launch(0, rblocks, ka, last(ka), buf[cur], 0, 0, nullptr);
      if (more) launch(bblocks, 0, 0, 0, buf[cur], na, last(na), buf[cur]);
    }
  }
  return check_launch("ssc_perturb_leapfrog");
}

template <int SK, int G, int RAD, int HS>
static int launch_perturb(const ssc_host_potential& hp, const ssc_sources& pert, const double* w0,
                          const double* dw0, const int32_t* start, int64_t n, double t0, double dt,
                          int nsteps, double* w_out, double* dw_out, hipStream_t st) {
  const int m = pert.n;
  int L = (m + G - 1) / G;
  int Lp = 1;
  while (Lp < L) Lp <<= 1;  // lanes per particle: a power of two dividing the block
  if (Lp > PT_BLOCK) return fail(SSC_E_LIMIT, "ssc_perturb_leapfrog: too many sources");
  const int ppb = PT_BLOCK / Lp;
  const size_t lds = SourceLDS<SK>::bytes(pert);
  if (lds > 60 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)perturb_kernel<SK, G, RAD, HS>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return fail(SSC_E_HIP, std::string("hipFuncSetAttribute: ") + hipGetErrorString(e));
  }
  const int64_t blocks = (n + ppb - 1) / ppb;
  hipLaunchKernelGGL((perturb_kernel<SK, G, RAD, HS>), dim3((unsigned)blocks), dim3(PT_BLOCK), lds, st,
                     hp, pert, w0, dw0, start, n, m, Lp, t0, dt, nsteps, w_out, dw_out);
  return check_launch("ssc_perturb_leapfrog");
}

}  // namespace ssc

using namespace ssc;

extern "C" int64_t ssc_perturb_workspace_bytes(int64_t n, int32_t nsteps) {
  if (n <= 0 || nsteps < 0) return 0;
  const int64_t per_row = n * PR_REC * 8;
  // two segments of at most 2 GiB each (1 GiB each: 200,000 particles x 16 sources, 2,000 steps
  // 9.3 ms for 8.7, a million x 8, 500 steps 13.8 for 10.9)
  const int64_t e = std::min(((int64_t)1 << 32) / per_row, perturb_rows_wanted(nsteps));
  return (e < 1 ? 1 : e) * per_row;
}

extern "C" int ssc_perturb_leapfrog(const ssc_host_potential* host, const ssc_sources* pert,
                                    const double* w0, const double* dw0, const int32_t* start_step,
                                    int64_t n, double t0, double dt, int32_t nsteps,
                                    int32_t with_radius, double* w_out, double* dw_out,
                                    void* workspace, int64_t workspace_bytes, void* stream) {
  int rc = validate_host(host);
  if (rc) return rc;
  if (!pert || pert->kind == SSC_SRC_NONE || pert->n <= 0)
    return fail(SSC_E_ARG, "ssc_perturb_leapfrog: needs at least one perturbing source");
  rc = validate_sources(pert, nsteps);
  if (rc) return rc;
  if (n < 0 || nsteps < 0) return fail(SSC_E_ARG, "ssc_perturb_leapfrog: negative size");
  if (n == 0) return SSC_OK;
  if (!w0 || !w_out || !dw_out) return fail(SSC_E_ARG, "ssc_perturb_leapfrog: NULL array");
  hipStream_t st = (hipStream_t)stream;
  const ssc_sources s = *pert;
  const int hs = host_signature(*host);
  int64_t E = 0;
  if (workspace) {
    E = perturb_segment_rows(n, nsteps, workspace_bytes);
    if (E < 1)
      return fail(SSC_E_ARG, "ssc_perturb_leapfrog: workspace smaller than one row of records (" +
                                 std::to_string(n * PR_REC * 8) + " bytes)");
    if (w_out == w0 || (dw0 && dw_out == dw0))
      return fail(SSC_E_ARG, "ssc_perturb_leapfrog: outputs must not alias the inputs");
  }
  const bool few = split_few(n, s.n, with_radius != 0);
#define SSC_PTS(K, G, R, H)                                                                      \
  launch_perturb_split<K, G, R, H>(*host, s, w0, dw0, start_step, n, t0, dt, nsteps, w_out,       \
                                   dw_out, (double*)workspace, E, st)
#define SSC_PT3(K, R, H)                                                                        \
  (E > 0 ? (few ? SSC_PTS(K, 2, R, H) : SSC_PTS(K, (R ? 4 : 8), R, H))                           \
         : launch_perturb<K, 8, R, H>(*host, s, w0, dw0, start_step, n, t0, dt, nsteps, w_out,  \
                                      dw_out, st))
#define SSC_PT(K, R)                                                                 \
  (hs == HS_MN_HQ_NFW ? SSC_PT3(K, R, HS_MN_HQ_NFW)                                  \
                      : (hs == HS_MN_HQ_HQ_NFW ? SSC_PT3(K, R, HS_MN_HQ_HQ_NFW)      \
                                               : SSC_PT3(K, R, HS_GENERIC)))
  if (with_radius) {
    switch (s.kind) {
      case SSC_SRC_STATIC: return SSC_PT(SSC_SRC_STATIC, 1);
      case SSC_SRC_TRACK: return SSC_PT(SSC_SRC_TRACK, 1);
      case SSC_SRC_LINE: return SSC_PT(SSC_SRC_LINE, 1);
      case SSC_SRC_LINE_HERNQUIST: return SSC_PT(SSC_SRC_LINE_HERNQUIST, 1);
    }
  } else {
    switch (s.kind) {
      case SSC_SRC_STATIC: return SSC_PT(SSC_SRC_STATIC, 0);
      case SSC_SRC_TRACK: return SSC_PT(SSC_SRC_TRACK, 0);
      case SSC_SRC_LINE: return SSC_PT(SSC_SRC_LINE, 0);
      case SSC_SRC_LINE_HERNQUIST: return SSC_PT(SSC_SRC_LINE_HERNQUIST, 0);
    }
  }
#undef SSC_PT
#undef SSC_PT3
#undef SSC_PTS
  return fail(SSC_E_ARG, "ssc_perturb_leapfrog: bad source kind");
}
