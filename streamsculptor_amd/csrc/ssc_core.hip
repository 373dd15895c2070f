// libssc_mi355x core: error plumbing, potential evaluation and the fixed-step leapfrog
// stream kernel (one particle per lane, FP64 state in VGPRs, Plummer source tables in LDS).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdio>
#include <cstring>
#include <string>
#include <type_traits>

#include "ssc_device.h"
#include "ssc_sources_lds.h"

namespace ssc {

static thread_local std::string g_last_error;

void set_error(const std::string& msg) { g_last_error = msg; }

int fail(int code, const std::string& msg) {
  g_last_error = msg;
  return code;
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return fail(SSC_E_LAUNCH, std::string(what) + ": kernel launch failed: " + hipGetErrorString(e));
  return SSC_OK;
}

int validate_host(const ssc_host_potential* host) {
  if (!host) return fail(SSC_E_ARG, "host potential descriptor is NULL");
  if (host->n_components < 0 || host->n_components > SSC_MAX_COMPONENTS)
    return fail(SSC_E_ARG, "host potential: n_components out of range [0, 8]");
  for (int c = 0; c < host->n_components; ++c) {
    const int k = host->c[c].kind;
    if (k < SSC_COMP_MIYAMOTO_NAGAI || k > SSC_COMP_PLUMMER)
      return fail(SSC_E_ARG, "host potential: unknown component kind " + std::to_string(k));
  }
  return SSC_OK;
}

int validate_sources(const ssc_sources* src, int32_t nsteps_needed, bool allow_groups) {
  if (!src || src->kind == SSC_SRC_NONE || src->n == 0) return SSC_OK;
  if (src->group_size != 0) {
    if (!allow_groups)
      return fail(SSC_E_ARG, "sources: grouped sources (group_size > 0) are only supported by "
                             "ssc_dopri5");
    if (src->group_size < 0 || src->group_size > SSC_MAX_SOURCES)
      return fail(SSC_E_LIMIT, "sources: group_size out of range [1, " +
                                   std::to_string(SSC_MAX_SOURCES) + "]");
    if (src->n < 0 || src->n % src->group_size != 0)
      return fail(SSC_E_ARG, "sources: n must be a multiple of group_size");
    if (!src->group) return fail(SSC_E_ARG, "sources: group_size > 0 needs the group array");
    if (src->kind != SSC_SRC_STATIC && src->kind != SSC_SRC_LINE &&
        src->kind != SSC_SRC_LINE_HERNQUIST)
      return fail(SSC_E_ARG, "sources: grouped sources must be STATIC, LINE or LINE_HERNQUIST");
  } else if (src->n < 0 || src->n > SSC_MAX_SOURCES) {
    return fail(SSC_E_LIMIT, "sources: n out of range [0, " + std::to_string(SSC_MAX_SOURCES) + "]");
  }
  if (!src->gm || !src->rs || !src->pos) return fail(SSC_E_ARG, "sources: NULL gm/rs/pos");
  if ((src->kind == SSC_SRC_TRACK || src->kind == SSC_SRC_TRACK_HERNQUIST) &&
      src->n_track < nsteps_needed + 1)
    return fail(SSC_E_ARG, "sources: TRACK table has " + std::to_string(src->n_track) +
                               " rows, the integration needs " + std::to_string(nsteps_needed + 1));
  if ((src->kind == SSC_SRC_LINE || src->kind == SSC_SRC_LINE_HERNQUIST) &&
      (!src->vel || !src->t0 || !src->t_window))
    return fail(SSC_E_ARG, "sources: LINE needs vel, t0 and t_window");
  if (src->kind < SSC_SRC_NONE || src->kind > SSC_SRC_TRACK_HERNQUIST)
    return fail(SSC_E_ARG, "sources: unknown kind " + std::to_string(src->kind));
  return SSC_OK;
}

static ssc_sources empty_sources() {
  ssc_sources s;
  memset(&s, 0, sizeof(s));
  return s;
}

// ------------------------------------------------------------------------------------------
// ssc_eval: G lanes per point (lane r takes sources r, r + G, ... and the group adds up), the
// sources staged EV_TILE at a time in LDS with their positions formed and r_s squared; only the
// outputs asked for (OUT: 1 phi, 2 gradient, 4 Hessian) are formed.  FP64 issue bound: a pair
// takes 13 instructions for phi, 18 for the gradient, 27 for the Hessian (six entries, the
// diagonal's common part summed apart).  262,144 points x 512 clumps, MI355X: phi 86 us, gradient
// 113 us, Hessian 153 us (a kernel that formed all nine Hessian entries for every call and read
// its sources from memory: 308 us for each of them).
// ------------------------------------------------------------------------------------------
constexpr int EV_BLOCK = 256, EV_TILE = 256;

// One source's share: phi, g[3], H[0, 1, 2, 4, 5, 8] without the diagonal's f, which fsum takes.
template <bool HQ, int OUT>
__device__ __forceinline__ void eval_pair(const SrcGeo& s, double gm, double x, double y, double z,
                                          double& phi, double* g, double* H, double& fsum) {
  const double dx = x - s.x, dy = y - s.y, dz = z - s.z;
  double f, k;
  if constexpr (HQ) {  // s.rs2 holds a: f = G m / (r (r + a)^2), k = -f (3 r + a) / (r^2 (r + a))
    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
    const double ir = rsq(r2);
    // at the centre, and where r^2 overflows, ir is NaN but the potential is not
    const double r = r2 > 0.0 && r2 < __builtin_inf() ? r2 * ir : r2;
    const double ia = div_patched(1.0, r + s.rs2);
    const double d1 = gm * ia * ia;
    f = d1 * ir;
    k = -(ir * ir) * fma(2.0 * d1, ia, f);
    if (OUT & 1) phi = fma(-gm, ia, phi);
  } else {
    // the operations of plummer_full, whose values the labels of the learned force keep
    const double is = rsq(dx * dx + dy * dy + dz * dz + s.rs2);
    f = gm * is * is * is;
    k = -3.0 * f * is * is;
    if (OUT & 1) phi -= gm * is;
  }
  if (OUT & 2) {
    g[0] = fma(f, dx, g[0]);
    g[1] = fma(f, dy, g[1]);
    g[2] = fma(f, dz, g[2]);
  }
  if (OUT & 4) {
    const double kx = k * dx, ky = k * dy, kz = k * dz;
    fsum += f;
    H[0] = fma(kx, dx, H[0]);
    H[1] = fma(kx, dy, H[1]);
    H[2] = fma(kx, dz, H[2]);
    H[4] = fma(ky, dy, H[4]);
    H[5] = fma(ky, dz, H[5]);
    H[8] = fma(kz, dz, H[8]);
  }
}

template <bool HQ, int G, int OUT>
__global__ __launch_bounds__(EV_BLOCK) void eval_kernel(ssc_host_potential hp, ssc_sources src,
                                                        const double* __restrict__ xyz, int64_t n,
                                                        double t, int step,
                                                        double* __restrict__ phi_out,
                                                        double* __restrict__ grad_out,
                                                        double* __restrict__ hess_out) {
  __shared__ SrcGeo geo[EV_TILE];
  __shared__ double gmv[EV_TILE];
  __shared__ int wave_count[EV_BLOCK / 64];
  const int r = threadIdx.x % G;
  const int64_t i = (int64_t)blockIdx.x * (EV_BLOCK / G) + threadIdx.x / G;
  const bool valid = i < n;
  double x = 1.0, y = 0.0, z = 0.0;
  if (valid) {
    x = xyz[3 * i];
    y = xyz[3 * i + 1];
    z = xyz[3 * i + 2];
  }
  // the sums start from the host's terms, on the group's first lane
  double sphi, sg[3], sH[9], fsum = 0.0;
  host_full(hp, x, y, z, sphi, sg, sH);
  if (G > 1 && r != 0) {
    sphi = sg[0] = sg[1] = sg[2] = 0.0;
#pragma unroll
    for (int q = 0; q < 9; ++q) sH[q] = 0.0;
  }
  const int m = src.kind == SSC_SRC_NONE ? 0 : src.n;
  for (int j0 = 0; j0 < m; j0 += EV_TILE) {
    // stage the tile's active sources in order (straight-line subhalos are active only inside
    // their windows; an inactive source is skipped, not added as zero)
    const int j = j0 + threadIdx.x;
    double sx = 0.0, sy = 0.0, sz = 0.0;
    const bool on = j < m && source_position(src, j, step, t, sx, sy, sz);
    const uint64_t mask = __ballot(on);
    const int w = threadIdx.x >> 6;
    __syncthreads();  // the previous tile has been read
    if ((threadIdx.x & 63) == 0) wave_count[w] = __popcll(mask);
    __syncthreads();
    int at = __popcll(mask & ((1ull << (threadIdx.x & 63)) - 1));
    for (int q = 0; q < w; ++q) at += wave_count[q];
    if (on) {
      const double rs = src.rs[j];
      geo[at] = SrcGeo{sx, sy, sz, HQ ? rs : rs * rs};
      gmv[at] = src.gm[j];
    }
    int cnt = 0;
#pragma unroll
    for (int q = 0; q < EV_BLOCK / 64; ++q) cnt += wave_count[q];
    __syncthreads();
#pragma unroll 4
    for (int q = r; q < cnt; q += G)
      eval_pair<HQ, OUT>(geo[q], gmv[q], x, y, z, sphi, sg, sH, fsum);
  }
  if (OUT & 1) sphi = group_sum<G>(sphi);
  if (OUT & 2)
#pragma unroll
    for (int c = 0; c < 3; ++c) sg[c] = group_sum<G>(sg[c]);
  if (OUT & 4) {
    fsum = group_sum<G>(fsum);
    sH[0] = group_sum<G>(sH[0]) + fsum;
    sH[1] = group_sum<G>(sH[1]);
    sH[2] = group_sum<G>(sH[2]);
    sH[4] = group_sum<G>(sH[4]) + fsum;
    sH[5] = group_sum<G>(sH[5]);
    sH[8] = group_sum<G>(sH[8]) + fsum;
  }
  if (!valid || r != 0) return;
  if ((OUT & 1) && phi_out) phi_out[i] = sphi;
  if ((OUT & 2) && grad_out) {
#pragma unroll
    for (int c = 0; c < 3; ++c) grad_out[3 * i + c] = sg[c];
  }
  if ((OUT & 4) && hess_out) {
    sH[3] = sH[1];
    sH[6] = sH[2];
    sH[7] = sH[5];
#pragma unroll
    for (int k = 0; k < 9; ++k) hess_out[9 * i + k] = sH[k];
  }
}

// Lanes per point: one when the points alone give four waves per SIMD; below that enough to
// spread a point's sources, at least four each, over otherwise idle lanes (a Hessian at 512
// clumps per call, 15 us of host time included: 1,000 points 16.9 us with 64 lanes and 40.6 us
// with one, 20,000 points 20.2 us with 16 and 40.8 us with one, 60,000 points 27.5 us with 4 and
// 28.5 us with one).
inline int eval_lanes(int64_t n, int nsrc) {
  int g = n >= 131072 ? 1 : (n >= 32768 ? 4 : (n >= 8192 ? 16 : 64));
  while (g > 1 && nsrc / g < 4) g >>= 2;
  return g;
}

template <bool HQ, int OUT>
static int launch_eval(const ssc_host_potential& hp, const ssc_sources& s, const double* xyz,
                       int64_t n, double t, int step, double* phi, double* grad, double* hess,
                       hipStream_t st) {
  const int g = eval_lanes(n, s.kind == SSC_SRC_NONE ? 0 : s.n);
  const unsigned blocks = (unsigned)((n * g + EV_BLOCK - 1) / EV_BLOCK);
#define SSC_EV(GV)                                                                              \
  hipLaunchKernelGGL((eval_kernel<HQ, GV, OUT>), dim3(blocks), dim3(EV_BLOCK), 0, st, hp, s, xyz, \
                     n, t, step, phi, grad, hess)
  switch (g) {
    case 4: SSC_EV(4); break;
    case 16: SSC_EV(16); break;
    case 64: SSC_EV(64); break;
    default: SSC_EV(1); break;
  }
#undef SSC_EV
  return check_launch("ssc_eval");
}

// ------------------------------------------------------------------------------------------
// Leapfrog: all lanes of a block walk the global grid together (k = block's earliest start ..
// nsteps-1); a particle kicks/drifts only once k >= its start.  Each lane carries P particles
// so that one LDS read of a source record serves P force terms.  Source tables live in LDS:
//   STATIC: rec[j] = (x, y, z, G*m), rs2[j]           (loaded once)
//   TRACK:  rows kb..kb+chunk of the trajectory table, rec[r][j] = (x, y, z, G*m)
//   LINE:   (x0, v, G*m, r_s^2, t0, t_window) per source, position formed per step
// add_grad(j0, js) sums sources j0, j0 + js, ... so a wave can also split one orbit's sum.
// ------------------------------------------------------------------------------------------
constexpr int LF_BLOCK = 256;

// Acceleration of P particles at grid row k / time t.
template <int SK, int P, int HS>
__device__ __forceinline__ void accel_P(const ssc_host_potential& hp, const SourceLDS<SK>& lds,
                                        int k, double t, const double* x, const double* y,
                                        const double* z, double* ax, double* ay, double* az) {
  double gx[P], gy[P], gz[P];
#pragma unroll
  for (int p = 0; p < P; ++p)
    host_grad_sig<HS, lean_host(SK)>(hp, x[p], y[p], z[p], gx[p], gy[p], gz[p]);
  lds.template add_grad<P>(k, t, x, y, z, gx, gy, gz, 0, 1);
#pragma unroll
  for (int p = 0; p < P; ++p) {
    ax[p] = -gx[p];
    ay[p] = -gy[p];
    az[p] = -gz[p];
  }
}

// The rows a launch saves, walked in order; the grid index of the save after the next is read a
// save ahead, so that no step waits for it.  One wave's step is a serial chain in which each
// branch and scalar instruction is seen, so the steps run in an inner loop up to the next saved
// row, which compares with nothing else; launches that save most of their steps (DENSE: the
// progenitors of streams) save inside the step instead, in straight code, because the way out of
// the inner loop and back costs 190 ns.  One orbit in the host, ns a step: not saved 296, saved
// every tenth step 391 -> 326 (inner loop), at every step 478 -> 390 (DENSE).
struct SaveRows {
  const int32_t* idx;
  int n, next, k, k_after;
  __device__ SaveRows(const int32_t* i, int nsave)
      : idx(i), n(nsave), next(0), k(at(0)), k_after(at(1)) {}
  __device__ int at(int j) const { return j < n ? idx[j] : INT_MIN; }  // none left
  __device__ bool up_to(int row) const { return next < n && k <= row; }
  __device__ bool due(int row) const { return k == row; }  // rows are >= 0
  // the row to step to from `row`: the next saved one, or the last
  __device__ int stop(int row, int last) const { return k > row && k < last ? k : last; }
  __device__ void advance() {
    ++next;
    k = k_after;
    k_after = at(next + 1);
  }
  // advance() if `hit`, without a branch (n > 0); the value read is first looked at a step later
  __device__ void advance_if(bool hit) {
    next += hit ? 1 : 0;
    k = hit ? (next < n ? k_after : INT_MIN) : k;
    k_after = idx[next + 1 < n ? next + 1 : n - 1];
  }
};

// The same walk for kernels whose step is long (many orbits among sources): the index is read
// where it is compared, and the step loop knows nothing of it (the two-level loop cost 3 to 7 %
// of a step of 12,500 to 100,000 orbits among 64 subhalos).
struct SaveScan {
  const int32_t* idx;
  int n, next;
  __device__ SaveScan(const int32_t* i, int nsave) : idx(i), n(nsave), next(0) {}
  __device__ bool up_to(int row) const { return next < n && idx[next] <= row; }
  __device__ bool due(int row) const { return next < n && idx[next] == row; }
  __device__ int stop(int row, int) const { return row + 1; }
  __device__ void advance() { ++next; }
};

template <int SK, int P, int HS, bool DENSE>
__global__ __launch_bounds__(LF_BLOCK) void leapfrog_kernel(
    ssc_host_potential hp, ssc_sources src, const double* __restrict__ w0,
    const int32_t* __restrict__ start, int64_t n, double t0, double dt, int nsteps,
    double* __restrict__ w_out, const int32_t* __restrict__ save_idx, int nsave,
    double* __restrict__ ys) {
  extern __shared__ __align__(16) char lds_raw[];
  __shared__ int kmin_sh;
  double x[P], y[P], z[P], vx[P], vy[P], vz[P], ax[P], ay[P], az[P];
  int s[P];
  int64_t idx[P];
  bool valid[P];
  int smin = nsteps;
#pragma unroll
  for (int p = 0; p < P; ++p) {
    idx[p] = (int64_t)blockIdx.x * (LF_BLOCK * P) + p * LF_BLOCK + threadIdx.x;
    valid[p] = idx[p] < n;
    s[p] = nsteps;
    x[p] = 1.0; y[p] = 0.0; z[p] = 0.0; vx[p] = vy[p] = vz[p] = 0.0;
    if (valid[p]) {
      int sp = start ? start[idx[p]] : 0;
      s[p] = sp < 0 ? 0 : (sp > nsteps ? nsteps : sp);
      const double* w = w0 + 6 * idx[p];
      x[p] = w[0]; y[p] = w[1]; z[p] = w[2]; vx[p] = w[3]; vy[p] = w[4]; vz[p] = w[5];
    }
    smin = min(smin, s[p]);
  }
  if (threadIdx.x == 0) kmin_sh = INT_MAX;
  __syncthreads();
  atomicMin(&kmin_sh, smin);
  SourceLDS<SK> lds;
  lds.init(src, lds_raw);
  __syncthreads();
  const int kmin = kmin_sh;
  // Save rows at grid indices <= kmin hold the initial state of every particle.
  typename std::conditional<SK == SSC_SRC_NONE, SaveRows, SaveScan>::type rows(save_idx, nsave);
  while (rows.up_to(kmin)) {
#pragma unroll
    for (int p = 0; p < P; ++p)
      if (valid[p]) {
        double* o = ys + ((int64_t)rows.next * n + idx[p]) * 6;
        o[0] = x[p]; o[1] = y[p]; o[2] = z[p]; o[3] = vx[p]; o[4] = vy[p]; o[5] = vz[p];
      }
    rows.advance();
  }
  const double h = 0.5 * dt;
  if (kmin < nsteps) {
    lds.stage(src, kmin, nsteps + 1);
    accel_P<SK, P, HS>(hp, lds, kmin, t0 + kmin * dt, x, y, z, ax, ay, az);
  }
  // A particle that has not started keeps its initial row; the force evaluated there at
  // t_{k+1} is exactly the initial force it needs when it starts at k + 1.
  double* o_next[P];  // DENSE: where the next saved row goes
  auto aim = [&]() {
#pragma unroll
    for (int p = 0; p < P; ++p) o_next[p] = ys + ((int64_t)rows.next * n + idx[p]) * 6;
  };
  if (DENSE) aim();
  for (int k = kmin; k < nsteps;) {
    const int stop = DENSE ? nsteps : rows.stop(k, nsteps);
    for (; k < stop; ++k) {
      lds.stage(src, k, nsteps + 1);
#pragma unroll
      for (int p = 0; p < P; ++p)
        if (k >= s[p]) {
          vx[p] = vx[p] + h * ax[p]; vy[p] = vy[p] + h * ay[p]; vz[p] = vz[p] + h * az[p];
          x[p] = x[p] + dt * vx[p]; y[p] = y[p] + dt * vy[p]; z[p] = z[p] + dt * vz[p];
        }
      accel_P<SK, P, HS>(hp, lds, k + 1, t0 + (k + 1) * dt, x, y, z, ax, ay, az);
#pragma unroll
      for (int p = 0; p < P; ++p)
        if (k >= s[p]) {
          vx[p] = vx[p] + h * ax[p]; vy[p] = vy[p] + h * ay[p]; vz[p] = vz[p] + h * az[p];
        }
      if constexpr (DENSE) {
        const bool hit = rows.k == k + 1;
#pragma unroll
        for (int p = 0; p < P; ++p)
          if (hit && valid[p]) {
            double* o = o_next[p];
            o[0] = x[p]; o[1] = y[p]; o[2] = z[p]; o[3] = vx[p]; o[4] = vy[p]; o[5] = vz[p];
          }
#pragma unroll
        for (int p = 0; p < P; ++p) o_next[p] += hit ? 6 * n : 0;
        rows.advance_if(hit);
        if (rows.k == k + 1) { ++k; break; }  // the same row again
      }
    }
    // block-uniform: every particle is now at grid index k (or holds its initial row)
    while (rows.due(k)) {
#pragma unroll
      for (int p = 0; p < P; ++p)
        if (valid[p]) {
          double* o = ys + ((int64_t)rows.next * n + idx[p]) * 6;
          o[0] = x[p]; o[1] = y[p]; o[2] = z[p]; o[3] = vx[p]; o[4] = vy[p]; o[5] = vz[p];
        }
      rows.advance();
      if (DENSE) aim();
    }
  }
#pragma unroll
  for (int p = 0; p < P; ++p)
    if (valid[p]) {
      double* o = w_out + 6 * idx[p];
      o[0] = x[p]; o[1] = y[p]; o[2] = z[p]; o[3] = vx[p]; o[4] = vy[p]; o[5] = vz[p];
    }
}

// G lanes per orbit: for batches too small to fill the chip one orbit per lane (1e5 particles
// are 1.5 waves per SIMD), G consecutive lanes split the orbit's source sum (lane r takes
// sources r, r + G, ...), combine it with a butterfly over the group and all carry the same
// orbit state.  Block-uniform grid walk and TRACK staging as in leapfrog_kernel.
template <int SK, int G, int HS>
__device__ __forceinline__ void accel_group(const ssc_host_potential& hp, const SourceLDS<SK>& lds,
                                            int k, double t, int r, double x, double y, double z,
                                            double& ax, double& ay, double& az) {
  double gx = 0.0, gy = 0.0, gz = 0.0;
  lds.template add_grad<1>(k, t, &x, &y, &z, &gx, &gy, &gz, r, G);
  gx = group_sum<G>(gx);
  gy = group_sum<G>(gy);
  gz = group_sum<G>(gz);
  double hx, hy, hz;
  host_grad_sig<HS, lean_host(SK)>(hp, x, y, z, hx, hy, hz);
  ax = -(hx + gx);
  ay = -(hy + gy);
  az = -(hz + gz);
}

template <int SK, int G, int HS>
__device__ __forceinline__ void leapfrog_group(
    const ssc_host_potential& hp, const ssc_sources& src, const double* __restrict__ w0,
    const int32_t* __restrict__ start, int64_t i, int64_t n, double t0, double dt, int nsteps,
    double* __restrict__ w_out, const int32_t* __restrict__ save_idx, int nsave,
    double* __restrict__ ys, char* lds_raw, int& kmin_sh) {
  const int r = threadIdx.x % G;
  const bool valid = i < n, lead = valid && r == 0;
  int s = nsteps;
  double x = 1.0, y = 0.0, z = 0.0, vx = 0.0, vy = 0.0, vz = 0.0;
  if (valid) {
    const int sp = start ? start[i] : 0;
    s = sp < 0 ? 0 : (sp > nsteps ? nsteps : sp);
    const double* w = w0 + 6 * i;
    x = w[0]; y = w[1]; z = w[2]; vx = w[3]; vy = w[4]; vz = w[5];
  }
  if (threadIdx.x == 0) kmin_sh = INT_MAX;
  __syncthreads();
  atomicMin(&kmin_sh, s);
  SourceLDS<SK> lds;
  lds.init(src, lds_raw);
  __syncthreads();
  const int kmin = kmin_sh;
  SaveScan rows(save_idx, nsave);
  while (rows.up_to(kmin)) {
    if (lead) {
      double* o = ys + ((int64_t)rows.next * n + i) * 6;
      o[0] = x; o[1] = y; o[2] = z; o[3] = vx; o[4] = vy; o[5] = vz;
    }
    rows.advance();
  }
  const double h = 0.5 * dt;
  double ax = 0.0, ay = 0.0, az = 0.0;
  if (kmin < nsteps) {
    lds.stage(src, kmin, nsteps + 1);
    accel_group<SK, G, HS>(hp, lds, kmin, t0 + kmin * dt, r, x, y, z, ax, ay, az);
  }
  for (int k = kmin; k < nsteps;) {
    const int stop = rows.stop(k, nsteps);
    for (; k < stop; ++k) {
      lds.stage(src, k, nsteps + 1);
      const bool act = k >= s;
      if (act) {
        vx = vx + h * ax; vy = vy + h * ay; vz = vz + h * az;
        x = x + dt * vx; y = y + dt * vy; z = z + dt * vz;
      }
      accel_group<SK, G, HS>(hp, lds, k + 1, t0 + (k + 1) * dt, r, x, y, z, ax, ay, az);
      if (act) {
        vx = vx + h * ax; vy = vy + h * ay; vz = vz + h * az;
      }
    }
    while (rows.due(k)) {
      if (lead) {
        double* o = ys + ((int64_t)rows.next * n + i) * 6;
        o[0] = x; o[1] = y; o[2] = z; o[3] = vx; o[4] = vy; o[5] = vz;
      }
      rows.advance();
    }
  }
  if (lead) {
    double* o = w_out + 6 * i;
    o[0] = x; o[1] = y; o[2] = z; o[3] = vx; o[4] = vy; o[5] = vz;
  }
}

// The first n_whole orbits (whole rounds of waves) take one lane each, the rest G lanes.
template <int SK, int G, int HS, bool WHOLE>
__global__ __launch_bounds__(LF_BLOCK) void leapfrog_group_kernel(
    ssc_host_potential hp, ssc_sources src, const double* __restrict__ w0,
    const int32_t* __restrict__ start, int64_t n_whole, int64_t n, double t0, double dt, int nsteps,
    double* __restrict__ w_out, const int32_t* __restrict__ save_idx, int nsave,
    double* __restrict__ ys) {
  extern __shared__ __align__(16) char lds_raw[];
  __shared__ int kmin_sh;
  const int64_t first = (int64_t)blockIdx.x * LF_BLOCK;
  if (WHOLE && first < n_whole)
    leapfrog_group<SK, 1, HS>(hp, src, w0, start, first + threadIdx.x, n, t0, dt, nsteps, w_out,
                              save_idx, nsave, ys, lds_raw, kmin_sh);
  else
    leapfrog_group<SK, G, HS>(hp, src, w0, start, n_whole + (first - n_whole + threadIdx.x) / G, n,
                              t0, dt, nsteps, w_out, save_idx, nsave, ys, lds_raw, kmin_sh);
}

// One wave per orbit: for a handful of orbits in a large source table (the progenitor in a
// clumpy halo) the 64 lanes split the source sum and combine it with a butterfly reduction;
// the orbit state is replicated in every lane.
constexpr int WAVE = 64;

template <int SK, int HS>
__device__ __forceinline__ void accel_wave(const ssc_host_potential& hp, const SourceLDS<SK>& lds,
                                           int k, double t, double x, double y, double z,
                                           double& ax, double& ay, double& az) {
  double gx = 0.0, gy = 0.0, gz = 0.0;
  lds.template add_grad<1>(k, t, &x, &y, &z, &gx, &gy, &gz, threadIdx.x, WAVE);
  gx = group_sum<WAVE>(gx);
  gy = group_sum<WAVE>(gy);
  gz = group_sum<WAVE>(gz);
  double hx, hy, hz;
  host_grad_sig<HS, lean_host(SK)>(hp, x, y, z, hx, hy, hz);
  ax = -(hx + gx);
  ay = -(hy + gy);
  az = -(hz + gz);
}

template <int SK, int HS, bool DENSE>
__global__ __launch_bounds__(WAVE) void leapfrog_wave_kernel(
    ssc_host_potential hp, ssc_sources src, const double* __restrict__ w0,
    const int32_t* __restrict__ start, int64_t n, double t0, double dt, int nsteps,
    double* __restrict__ w_out, const int32_t* __restrict__ save_idx, int nsave,
    double* __restrict__ ys) {
  extern __shared__ __align__(16) char lds_raw[];
  const int64_t i = blockIdx.x;
  const bool lead = threadIdx.x == 0;
  int s = start ? start[i] : 0;
  s = s < 0 ? 0 : (s > nsteps ? nsteps : s);
  const double* w = w0 + 6 * i;
  double x = w[0], y = w[1], z = w[2], vx = w[3], vy = w[4], vz = w[5];
  SourceLDS<SK> lds;
  lds.init(src, lds_raw);
  __syncthreads();
  SaveRows rows(save_idx, nsave);
  while (rows.up_to(s)) {
    if (lead) {
      double* o = ys + ((int64_t)rows.next * n + i) * 6;
      o[0] = x; o[1] = y; o[2] = z; o[3] = vx; o[4] = vy; o[5] = vz;
    }
    rows.advance();
  }
  const double h = 0.5 * dt;
  double ax = 0, ay = 0, az = 0;
  if (s < nsteps) {
    lds.template stage<8>(src, s, nsteps + 1);
    accel_wave<SK, HS>(hp, lds, s, t0 + s * dt, x, y, z, ax, ay, az);
  }
  double* o_next = ys + ((int64_t)rows.next * n + i) * 6;  // DENSE: where the next saved row goes
  for (int k = s; k < nsteps;) {
    const int stop = DENSE ? nsteps : rows.stop(k, nsteps);
    for (; k < stop; ++k) {
      lds.template stage<8>(src, k, nsteps + 1);
      vx = vx + h * ax; vy = vy + h * ay; vz = vz + h * az;
      x = x + dt * vx; y = y + dt * vy; z = z + dt * vz;
      accel_wave<SK, HS>(hp, lds, k + 1, t0 + (k + 1) * dt, x, y, z, ax, ay, az);
      vx = vx + h * ax; vy = vy + h * ay; vz = vz + h * az;
      if (DENSE) {
        const bool hit = rows.k == k + 1;
        if (hit && lead) {
          double* o = o_next;
          o[0] = x; o[1] = y; o[2] = z; o[3] = vx; o[4] = vy; o[5] = vz;
        }
        o_next += hit ? 6 * n : 0;
        rows.advance_if(hit);
        if (rows.k == k + 1) { ++k; break; }  // the same row again
      }
    }
    while (rows.due(k)) {
      if (lead) {
        double* o = ys + ((int64_t)rows.next * n + i) * 6;
        o[0] = x; o[1] = y; o[2] = z; o[3] = vx; o[4] = vy; o[5] = vz;
      }
      rows.advance();
      o_next += 6 * n;
    }
  }
  if (lead) {
    double* o = w_out + 6 * i;
    o[0] = x; o[1] = y; o[2] = z; o[3] = vx; o[4] = vy; o[5] = vz;
  }
}

// Orbits in the analytic host alone, for batches too small to fill the chip, where the step's
// latency sets the rate: the host components are spread over the waves of a block (wave c forms
// component c's gradient for the block's 64 orbits, one per lane; the kinds differ, so lanes of
// one wave could not share the work without running every kind's code), the waves exchange
// their gradient parts through LDS and each accumulates them in component order with the
// operations of host_grad (so the orbits are bit-identical to the one-lane kernels') and
// advances the same orbits.  One barrier per force evaluation (parts double-buffered).
__global__ __launch_bounds__(WAVE * SSC_MAX_COMPONENTS) void leapfrog_comp_kernel(
    ssc_host_potential hp, const double* __restrict__ w0, const int32_t* __restrict__ start,
    int64_t n, double t0, double dt, int nsteps, double* __restrict__ w_out,
    const int32_t* __restrict__ save_idx, int nsave, double* __restrict__ ys) {
  __shared__ double part[2][SSC_MAX_COMPONENTS][WAVE][3];  // f, zm, zadd of each component
  __shared__ int kmin_sh;
  const int l = threadIdx.x & (WAVE - 1), c = threadIdx.x / WAVE;
  const int64_t i = (int64_t)blockIdx.x * WAVE + l;
  const bool valid = i < n;
  const bool writer = valid && c == 0;
  double x = 1.0, y = 0.0, z = 0.0, vx = 0.0, vy = 0.0, vz = 0.0;
  int s = nsteps;
  if (valid) {
    const double* w = w0 + 6 * i;
    x = w[0]; y = w[1]; z = w[2]; vx = w[3]; vy = w[4]; vz = w[5];
    const int sp = start ? start[i] : 0;
    s = sp < 0 ? 0 : (sp > nsteps ? nsteps : sp);
  }
  if (threadIdx.x == 0) kmin_sh = INT_MAX;
  __syncthreads();
  atomicMin(&kmin_sh, s);
  __syncthreads();
  const int kmin = kmin_sh;
  const int nc = hp.n_components;
  int buf = 0;
  // block-uniform: every thread calls it the same number of times
  auto accel = [&](double& ax, double& ay, double& az) {
    double f, zm;
    bool zadd;
    comp_grad_parts(hp.c[c], x, y, z, f, zm, zadd);
    part[buf][c][l][0] = f; part[buf][c][l][1] = zm; part[buf][c][l][2] = zadd ? 1.0 : 0.0;
    __syncthreads();
    double gx = 0.0, gy = 0.0, gz = 0.0;
    for (int q = 0; q < nc; ++q)
      comp_grad_add(part[buf][q][l][0], part[buf][q][l][1], part[buf][q][l][2] != 0.0, x, y, z,
                    gx, gy, gz);
    ax = -gx; ay = -gy; az = -gz;
    buf ^= 1;
  };
  SaveRows rows(save_idx, nsave);
  while (rows.up_to(kmin)) {
    if (writer) {
      double* o = ys + ((int64_t)rows.next * n + i) * 6;
      o[0] = x; o[1] = y; o[2] = z; o[3] = vx; o[4] = vy; o[5] = vz;
    }
    rows.advance();
  }
  const double h = 0.5 * dt;
  double ax = 0.0, ay = 0.0, az = 0.0;
  if (kmin < nsteps) accel(ax, ay, az);
  // A particle that has not started keeps its initial row; the force evaluated there is the
  // initial force it needs when it starts.
  for (int k = kmin; k < nsteps;) {
    const int stop = rows.stop(k, nsteps);
    for (; k < stop; ++k) {
      const bool act = k >= s;
      if (act) {
        vx = vx + h * ax; vy = vy + h * ay; vz = vz + h * az;
        x = x + dt * vx; y = y + dt * vy; z = z + dt * vz;
      }
      accel(ax, ay, az);
      if (act) {
        vx = vx + h * ax; vy = vy + h * ay; vz = vz + h * az;
      }
    }
    while (rows.due(k)) {
      if (writer) {
        double* o = ys + ((int64_t)rows.next * n + i) * 6;
        o[0] = x; o[1] = y; o[2] = z; o[3] = vx; o[4] = vy; o[5] = vz;
      }
      rows.advance();
    }
  }
  if (writer) {
    double* o = w_out + 6 * i;
    o[0] = x; o[1] = y; o[2] = z; o[3] = vx; o[4] = vy; o[5] = vz;
  }
}

static int set_lds(const void* fn, size_t lds) {
  if (lds > 160 * 1024) return fail(SSC_E_LIMIT, "ssc_leapfrog: source table exceeds LDS");
  if (lds > 60 * 1024) {
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return fail(SSC_E_HIP, std::string("hipFuncSetAttribute: ") + hipGetErrorString(e));
  }
  return SSC_OK;
}

// Most orbits that take a wave each.  Every orbit has a SIMD of its own (512 clumps: 1,000 orbits
// 1.81 us a step against 2.87 with 16 lanes an orbit, 2,000 orbits 4.39 against 2.96; one orbit in 20
// tracked subhalos saved at every step 0.85 against 1.12, in 4 clumps 0.74 unsaved against 0.70: from
// 8 sources on).  Up to two or so to a SIMD for orbits that start all along the grid among many
// sources, half of whose waves wait for nobody's earlier start (1,300 orbits, 100 rows: 256 clumps
// 0.113 ms against 0.166 with 16 lanes an orbit, 512 clumps 0.136 against 0.242; 2,500 among 512
// 0.195 against 0.243, but among 1,024 0.451 against 0.393; 1,300 among 64 0.105 against 0.110).  Twice
// as many with straight-line sources, whose chains leave a SIMD idle (60 rows: 1,500 orbits, 200
// Hernquist subhalos 0.134 ms against 0.204, ragged 3,000 0.137 against 0.197).
static int64_t wave_orbits(int nsrc, bool ragged, bool line) {
  if (line) return (nsrc < 64 ? 1024 : 2048) * (ragged ? 2 : 1);
  if (!ragged || nsrc < 64) return 1024;
  return nsrc >= 256 && nsrc <= 512 ? 2560 : std::min(2048, 768 + 10 * nsrc);
}

// Launch shape: a wave per orbit (see wave_orbits); two particles per lane for batches that fill
// the chip several times over, unless the pairing costs a round of waves (512 clumps: 1e6 orbits
// 326 us against 331, 4e5 169 against 153), which pays all the same where two particles share the
// place of a straight-line source (200 Hernquist subhalos, 8e5 orbits, 60 rows 10.5 ms against
// 11.6); group_lanes otherwise.  Without sources: for up to
// 65536 orbits in a host of no known signature, host components over waves; one particle per lane
// otherwise (with straight-line host code for the known hosts, which is faster still).
template <int SK, int HS>
static int launch_leapfrog(const ssc_host_potential& hp, const ssc_sources& src, const double* w0,
                           const int32_t* start, int64_t n, double t0, double dt, int nsteps,
                           double* w_out, const int32_t* save_idx, int nsave, double* ys, bool ragged,
                           hipStream_t st) {
  const size_t lds = SourceLDS<SK>::bytes(src);
  const bool dense = nsave > nsteps / 2;  // see SaveRows
  constexpr bool LINE = SK == SSC_SRC_LINE || SK == SSC_SRC_LINE_HERNQUIST;
  const int64_t waves = wave_orbits(src.n, ragged, LINE);
  if (SK != SSC_SRC_NONE && src.n >= 8 && n <= waves) {
    auto kernel = dense ? leapfrog_wave_kernel<SK, HS, true> : leapfrog_wave_kernel<SK, HS, false>;
    int rc = set_lds((const void*)kernel, lds);
    if (rc) return rc;
    hipLaunchKernelGGL(kernel, dim3((unsigned)n), dim3(WAVE), lds, st, hp, src, w0,
                       start, n, t0, dt, nsteps, w_out, save_idx, nsave, ys);
    return check_launch("ssc_leapfrog");
  }
  if (SK != SSC_SRC_NONE && src.n >= 16 && n >= 393216 &&
      (LINE || 2 * ((n + 131071) / 131072) <= (n + 65535) / 65536)) {
    int rc = set_lds((const void*)leapfrog_kernel<SK, 2, HS, false>, lds);
    if (rc) return rc;
    const int64_t blocks = (n + 2 * LF_BLOCK - 1) / (2 * LF_BLOCK);
    hipLaunchKernelGGL((leapfrog_kernel<SK, 2, HS, false>), dim3((unsigned)blocks), dim3(LF_BLOCK), lds, st,
                       hp, src, w0, start, n, t0, dt, nsteps, w_out, save_idx, nsave, ys);
    return check_launch("ssc_leapfrog");
  }
  if (SK == SSC_SRC_NONE && HS == HS_GENERIC && hp.n_components >= 2 && n <= 65536) {
    const int64_t blocks = (n + WAVE - 1) / WAVE;
    hipLaunchKernelGGL(leapfrog_comp_kernel, dim3((unsigned)blocks),
                       dim3(WAVE * hp.n_components), 0, st, hp, w0, start, n, t0, dt, nsteps,
                       w_out, save_idx, nsave, ys);
    return check_launch("ssc_leapfrog");
  }
  int64_t n_whole = 0;
  const int g = SK == SSC_SRC_NONE ? 1
                : LINE             ? group_lanes_line(n, src.n, ragged, &n_whole)
                                   : group_lanes(n, src.n, ragged, &n_whole);
#define SSC_GROUP(GV)                                                                              \
  if (g == GV) {                                                                                   \
    auto kernel = n_whole ? leapfrog_group_kernel<SK, GV, HS, true>                                \
                          : leapfrog_group_kernel<SK, GV, HS, false>;                              \
    int rc = set_lds((const void*)kernel, lds);                                                    \
    if (rc) return rc;                                                                             \
    const int64_t blocks = n_whole / LF_BLOCK + (n - n_whole + LF_BLOCK / GV - 1) / (LF_BLOCK / GV); \
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(LF_BLOCK), lds, st, hp, src, w0, start, \
                       n_whole, n, t0, dt, nsteps, w_out, save_idx, nsave, ys);                    \
    return check_launch("ssc_leapfrog");                                                           \
  }
  SSC_GROUP(2)
  SSC_GROUP(4)
  SSC_GROUP(8)
  SSC_GROUP(16)
#undef SSC_GROUP
  auto kernel = SK == SSC_SRC_NONE && dense ? leapfrog_kernel<SK, 1, HS, SK == SSC_SRC_NONE>
                                            : leapfrog_kernel<SK, 1, HS, false>;
  int rc = set_lds((const void*)kernel, lds);
  if (rc) return rc;
  const int64_t blocks = (n + LF_BLOCK - 1) / LF_BLOCK;
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(LF_BLOCK), lds, st, hp, src, w0, start, n,
                     t0, dt, nsteps, w_out, save_idx, nsave, ys);
  return check_launch("ssc_leapfrog");
}

}  // namespace ssc

using namespace ssc;

// ssc_leapfrog; `ragged`: the orbits start all along the grid (chooses the lanes per orbit only).
static int leapfrog_run(const ssc_host_potential* host, const ssc_sources* src, const double* w0,
                        const int32_t* start_step, int64_t n, double t0, double dt,
                        int32_t nsteps, double* w_out, const int32_t* save_idx, int32_t nsave,
                        double* ys, bool ragged, void* stream) {
  int rc = validate_host(host);
  if (rc) return rc;
  if (n < 0 || nsteps < 0 || nsave < 0) return fail(SSC_E_ARG, "ssc_leapfrog: negative size");
  if (n == 0) return SSC_OK;
  if (!w0 || !w_out) return fail(SSC_E_ARG, "ssc_leapfrog: w0 or w_out is NULL");
  if (nsave > 0 && (!save_idx || !ys)) return fail(SSC_E_ARG, "ssc_leapfrog: nsave > 0 needs save_idx and ys");
  if (nsave == 0) { save_idx = nullptr; ys = nullptr; }
  if ((n + LF_BLOCK - 1) / LF_BLOCK > (int64_t)INT_MAX)
    return fail(SSC_E_LIMIT, "ssc_leapfrog: too many particles");
  rc = validate_sources(src, nsteps);
  if (rc) return rc;
  ssc_sources s = src ? *src : empty_sources();
  if (s.n == 0) s.kind = SSC_SRC_NONE;
  hipStream_t st = (hipStream_t)stream;
  const int hs = host_signature(*host);
#define SSC_LF3(K, H) launch_leapfrog<K, H>(*host, s, w0, start_step, n, t0, dt, nsteps, w_out, save_idx, nsave, ys, ragged, st)
#define SSC_LF(K)                                                                                 \
  (hs == HS_MN_HQ_NFW ? SSC_LF3(K, HS_MN_HQ_NFW)                                                 \
                      : (hs == HS_MN_HQ_HQ_NFW ? SSC_LF3(K, HS_MN_HQ_HQ_NFW) : SSC_LF3(K, HS_GENERIC)))
  switch (s.kind) {
    case SSC_SRC_NONE: return SSC_LF(SSC_SRC_NONE);
    case SSC_SRC_STATIC: return SSC_LF(SSC_SRC_STATIC);
    case SSC_SRC_TRACK: return SSC_LF(SSC_SRC_TRACK);
    case SSC_SRC_LINE: return SSC_LF(SSC_SRC_LINE);
    case SSC_SRC_LINE_HERNQUIST: return SSC_LF(SSC_SRC_LINE_HERNQUIST);
    case SSC_SRC_TRACK_HERNQUIST: return SSC_LF(SSC_SRC_TRACK_HERNQUIST);
    default: return fail(SSC_E_ARG, "ssc_leapfrog: bad source kind");
  }
#undef SSC_LF
#undef SSC_LF3
}

extern "C" {

const char* ssc_last_error(void) { return g_last_error.c_str(); }

const char* ssc_version(void) { return "libssc_mi355x 0.1 (gfx950)"; }

int ssc_eval(const ssc_host_potential* host, const ssc_sources* src, const double* xyz, int64_t n,
             double t, int32_t step, double* phi, double* grad, double* hess, void* stream) {
  int rc = validate_host(host);
  if (rc) return rc;
  if (n < 0) return fail(SSC_E_ARG, "ssc_eval: n < 0");
  if (n == 0) return SSC_OK;
  if (!xyz) return fail(SSC_E_ARG, "ssc_eval: xyz is NULL");
  rc = validate_sources(src, step < 0 ? 0 : step);
  if (rc) return rc;
  ssc_sources s = src ? *src : empty_sources();
  if (s.n == 0) s.kind = SSC_SRC_NONE;
  if ((n + EV_BLOCK - 1) / EV_BLOCK > (int64_t)INT_MAX)
    return fail(SSC_E_LIMIT, "ssc_eval: too many points");
  const bool hq = s.kind == SSC_SRC_LINE_HERNQUIST || s.kind == SSC_SRC_TRACK_HERNQUIST;
  const int out = (phi ? 1 : 0) | (grad ? 2 : 0) | (hess ? 4 : 0);
  hipStream_t st = (hipStream_t)stream;
#define SSC_EVAL(O)                                                               \
  (hq ? launch_eval<true, O>(*host, s, xyz, n, t, step, phi, grad, hess, st)       \
      : launch_eval<false, O>(*host, s, xyz, n, t, step, phi, grad, hess, st))
  switch (out) {
    case 0: return SSC_OK;
    case 1: return SSC_EVAL(1);
    case 2: return SSC_EVAL(2);
    case 3: return SSC_EVAL(3);
    case 4: return SSC_EVAL(4);
    default: return SSC_EVAL(7);
  }
#undef SSC_EVAL
}

int ssc_leapfrog(const ssc_host_potential* host, const ssc_sources* src, const double* w0,
                 const int32_t* start_step, int64_t n, double t0, double dt, int32_t nsteps,
                 double* w_out, const int32_t* save_idx, int32_t nsave, double* ys,
                 void* stream) {
  return leapfrog_run(host, src, w0, start_step, n, t0, dt, nsteps, w_out, save_idx, nsave, ys,
                      start_step != nullptr, stream);
}

int ssc_leapfrog_window(const ssc_host_potential* host, const ssc_sources* src, const double* w0,
                        const int32_t* start_step, int64_t n, double t0, double dt,
                        int32_t nsteps, double* w_out, void* stream) {
  return leapfrog_run(host, src, w0, start_step, n, t0, dt, nsteps, w_out, nullptr, 0, nullptr,
                      false, stream);
}

}  // extern "C"
