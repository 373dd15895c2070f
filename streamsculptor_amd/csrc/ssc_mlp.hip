// The clump-force MLP on gfx950: BF16 MFMA training (forward, backward, Adam) and the packed,
// register-chained inference form.
//
// Network: 3 -> 256 -> 256 -> 256 -> 4, SiLU after the three hidden layers.  Master parameters
// are fp32; every matrix product runs on v_mfma_f32_32x32x16_bf16 with BF16 operands (weights
// and activations rounded to nearest-even) and fp32 accumulation.  The 3-wide first layer runs
// on the fp32 VALU (BF16-rounded weights, fp32 inputs) so the input coordinates keep fp32
// resolution.
//
// Training path: 64x64 block tiles of four 32x32 wave tiles, split-K for the batch reductions of
// the weight gradients, several jobs per launch.
// Inference path: weights pre-packed in MFMA fragment order; a wave evaluates 16 points per
// tile with the activations kept in registers between layers (points on the MFMA N axis).
#include <hip/hip_runtime.h>

#include <cstring>
#include <string>

#include "ssc_device.h"
#include "ssc_mlp.h"
#include "ssc_mlp_tile.h"

namespace ssc {
namespace mlp {

// ------------------------------------------------------------------------------------------
// Training kernels.  A minibatch's matrix products are small (8192 x 256 x 256: 1 GFLOP, 12 MB),
// so an iteration is bound by launches, load latency and how many blocks each launch has.  One
// launch therefore carries every job whose inputs are ready (ProductJobs, FinishJobs: products,
// column sums and reductions side by side, a block range each); a product's epilogue applies the
// activation or its derivative; and a product's tile loads its whole K range (up to TK) into LDS
// with every load in flight at once.  Operands are kept K-contiguous for all products: activations and
// their gradients are written in both orders by the epilogue that forms them.  Every sum that a
// gradient goes through keeps its order (K ascending in steps of 16 within a tile, the split-K
// chunks, the column sums), so a training run gives the same network bit for bit; the loss, which
// nothing but the caller reads, is added up by tiles of 64 points, and its last bit is not that of
// sums over 256.  An iteration of 8,192 points (loss, gradients, Adam): 31 launches and 281 us with
// a kernel per step and a 32-wide K stage, 11 launches and 127 us now; of it 21 us per backward
// launch (its 20 MB would take 5), 12 us per forward product, 14 us the first layer's gradient
// (chains of 128 additions, the order's price).
//
// A product: C(m, n) = sum_k A(m, k) B(n, k), A(m, k) = a[m * sa + k * ka] and B likewise, in
// 64 x 64 tiles by four waves of 32 x 32; K split into chunks of kchunk.
// ------------------------------------------------------------------------------------------
constexpr int GT = 64;     // block tile
constexpr int GK = 32;     // granularity of the split-K chunks
constexpr int TK = 256;    // k's staged at once
constexpr int TPAD = 264;  // LDS row pitch (elements): 16-byte fragments, rows 4 banks apart
constexpr int CS_ROWS = 512;  // batch rows per partial of the column sums

enum { EPI_PART, EPI_ACT, EPI_DACT, EPI_OUT };
struct Operand {
  const uint16_t* p;
  int64_t s, k;  // strides of row and k; 16-byte loads when k == 1 and s % 8 == 0
  int rows;
};
struct Product {
  Operand a, b;
  int K, kchunk, tm, tn;
  int epi;
  const float* bias;     // EPI_ACT, EPI_OUT
  const float* Z;        // EPI_DACT: pre-activations [m][256]
  float* out;            // PART: [z][M][N]; ACT: Z; DACT: dZ; OUT: y
  uint16_t* out16;       // ACT: silu(Z); DACT: dZ; OUT: dY, row major (may be NULL)
  uint16_t* out16t;      // the same transposed, row pitch ldt (may be NULL)
  int64_t ldt;
  // EPI_OUT with a loss (target != NULL): dY = 2 w (y - t) / sum w, block partials of the loss
  const float *target, *weight, *wsum_dev;
  float inv_wsum;
  float *dY, *loss_part;
};
struct ColSum {  // partial column sums of D [nb][ncol]
  const float* D;
  float* part;
  int64_t nb;
  int ncol;
};
struct Layer1Grad {  // partials of dW1, db1
  const float *dZ, *x;
  float* part;
  int64_t nb;
};
struct Reduce {  // out[e] = sum_z part[z][e]
  const float* part;
  float* out;
  int nz, ne;
};

struct alignas(16) TileLds {
  uint16_t a[GT][TPAD], b[GT][TPAD];
};

// One operand's 64 rows x TK k's of a stage: 16-byte pieces, all eight of a thread's loads in
// flight before its first LDS store, zeros past the edges.  Pieces need K contiguous, rows of a
// multiple of 8 elements and a K range that ends on a piece; other operands (the four-wide output
// gradient and weights, a ragged batch's last stage) are read element by element.
constexpr int NPIECE = TK / 8 * GT / 256;
__device__ __forceinline__ bool in_pieces(const Operand& o, int k0, int ke) {
  return o.k == 1 && (o.s & 7) == 0 && (ke - k0 >= TK || ((ke - k0) & 7) == 0);
}
__device__ __forceinline__ void load_pieces(const Operand& o, int r0, int k0, int ke, int t,
                                            uint4 (&v)[NPIECE]) {
  const int kc = k0 + ((t & 31) << 3);
#pragma unroll
  for (int u = 0; u < NPIECE; ++u) {
    const int r = r0 + (t >> 5) + 8 * u;
    v[u] = make_uint4(0, 0, 0, 0);
    if (r < o.rows && kc < ke) v[u] = *reinterpret_cast<const uint4*>(o.p + (int64_t)r * o.s + kc);
  }
}
__device__ __forceinline__ void store_pieces(uint16_t (*X)[TPAD], int t,
                                             const uint4 (&v)[NPIECE]) {
#pragma unroll
  for (int u = 0; u < NPIECE; ++u)
    *reinterpret_cast<uint4*>(&X[(t >> 5) + 8 * u][(t & 31) << 3]) = v[u];
}
__device__ __forceinline__ void fill_elements(const Operand& o, int r0, int k0, int ke, int kw,
                                              int t, uint16_t (*X)[TPAD]) {
  for (int c = t; c < GT * kw; c += 256) {
    // neighbouring threads along the contiguous direction
    const int row = o.k == 1 ? c / kw : c % GT, kk = o.k == 1 ? c - row * kw : c / GT;
    const int r = r0 + row, k = k0 + kk;
    X[row][kk] = r < o.rows && k < ke ? o.p[(int64_t)r * o.s + (int64_t)k * o.k] : (uint16_t)0;
  }
}

template <int EPI>
__device__ __forceinline__ void product(const Product& g, int blk, TileLds& lds) {
  const int mi = blk % g.tm, ni = (blk / g.tm) % g.tn, z = blk / (g.tm * g.tn);
  const int m0 = mi * GT, n0 = ni * GT;
  const int kb = z * g.kchunk, ke = min(g.K, kb + g.kchunk);
  const int t = threadIdx.x, l = t & 63, w = t >> 6;
  const int wm = w & 1, wn = w >> 1;
  f32x16 acc = {};
  for (int k0 = kb; k0 < ke; k0 += TK) {
    const int kw = min(TK, (ke - k0 + 15) & ~15);
    const bool pa = in_pieces(g.a, k0, ke), pb = in_pieces(g.b, k0, ke);
    uint4 va[NPIECE], vb[NPIECE];
    if (pa) load_pieces(g.a, m0, k0, ke, t, va);
    if (pb) load_pieces(g.b, n0, k0, ke, t, vb);
    if (k0 > kb) __syncthreads();  // the previous stage has been read
    if (pa)
      store_pieces(lds.a, t, va);
    else
      fill_elements(g.a, m0, k0, ke, kw, t, lds.a);
    if (pb)
      store_pieces(lds.b, t, vb);
    else
      fill_elements(g.b, n0, k0, ke, kw, t, lds.b);
    __syncthreads();
#pragma unroll 4
    for (int ks = 0; ks < kw; ks += 16) {
      const bf16x8 a =
          *reinterpret_cast<const bf16x8*>(&lds.a[32 * wm + (l & 31)][ks + 8 * (l >> 5)]);
      const bf16x8 b =
          *reinterpret_cast<const bf16x8*>(&lds.b[32 * wn + (l & 31)][ks + 8 * (l >> 5)]);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
    }
  }
  const int M = g.a.rows, N = g.b.rows;
  const int col = n0 + 32 * wn + (l & 31);
  const float bv = g.bias && col < N ? g.bias[col] : 0.0f;
  float inv = g.inv_wsum, lsum = 0.0f;
  if (EPI == EPI_OUT && g.target && g.wsum_dev) inv = 1.0f / *g.wsum_dev;
#pragma unroll
  for (int q = 0; q < 4; ++q) {  // rows row0 .. row0 + 3 of this lane's column
    const int row0 = m0 + 32 * wm + 8 * q + 4 * (l >> 5);
    uint16_t h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = row0 + e;
      const bool in = row < M && col < N;
      const float c = acc[4 * q + e] + bv;
      h[e] = 0;
      if (!in) continue;
      if constexpr (EPI == EPI_PART) {
        g.out[((int64_t)z * M + row) * N + col] = c;
      } else if constexpr (EPI == EPI_ACT) {
        g.out[(int64_t)row * H + col] = c;
        h[e] = f2bf(silu(c));
        g.out16[(int64_t)row * H + col] = h[e];
      } else if constexpr (EPI == EPI_DACT) {
        const float d = c * silu_grad(g.Z[(int64_t)row * H + col]);
        g.out[(int64_t)row * H + col] = d;
        h[e] = f2bf(d);
        if (g.out16) g.out16[(int64_t)row * H + col] = h[e];
      } else {
        g.out[(int64_t)row * OUT + col] = c;
        if (g.target) {
          const float wt = g.weight ? g.weight[row] : 1.0f;
          const float d = c - g.target[(int64_t)row * OUT + col];
          lsum += wt * d * d;
          const float gr = 2.0f * wt * d * inv;
          g.dY[(int64_t)row * OUT + col] = gr;
          h[e] = f2bf(gr);
          g.out16[(int64_t)row * OUT + col] = h[e];
        }
      }
    }
    if (EPI != EPI_PART && g.out16t && col < N) {
      uint16_t* o = g.out16t + (int64_t)col * g.ldt + row0;
      if (row0 + 4 <= M) {
        uint2 v;
        memcpy(&v, h, 8);
        *reinterpret_cast<uint2*>(o) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (row0 + e < M) o[e] = h[e];
      }
    }
  }
  if (EPI == EPI_OUT && g.target) {
    float* red = reinterpret_cast<float*>(&lds);
    __syncthreads();  // the tiles have been read
    red[t] = lsum * inv;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
      if (t < s) red[t] += red[t + s];
      __syncthreads();
    }
    if (t == 0) g.loss_part[mi] = red[0];
  }
}

// Column sums over the batch in two deterministic passes: blocks of (64 columns x 4 row
// phases) over batch chunks of CS_ROWS rows write partials, a later job adds the chunks.
__device__ void col_sum(const ColSum& g, int blk, TileLds& lds) {
  float(*red)[64] = reinterpret_cast<float(*)[64]>(&lds);
  const int nc = (g.ncol + 63) / 64, by = blk / nc;
  const int c = (blk - by * nc) * 64 + (threadIdx.x & 63), ph = threadIdx.x >> 6;
  const int64_t b0 = (int64_t)by * CS_ROWS, b1 = min(g.nb, b0 + CS_ROWS);
  float s = 0.0f;
  if (c < g.ncol)
    // rows b0 + ph, b0 + ph + 4, ... added in order; the loads of 32 of them are issued first
    for (int64_t b = b0 + ph; b < b1; b += 128) {
      float v[32];
#pragma unroll
      for (int u = 0; u < 32; ++u) v[u] = b + 4 * u < b1 ? g.D[(b + 4 * u) * g.ncol + c] : 0.0f;
#pragma unroll
      for (int u = 0; u < 32; ++u)
        if (b + 4 * u < b1) s += v[u];
    }
  red[ph][threadIdx.x & 63] = s;
  __syncthreads();
  if (ph == 0 && c < g.ncol)
    g.part[(int64_t)by * g.ncol + c] =
        red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
}

// dW1[o][i] = sum_b dZ1[b][o] x[b][i] and db1[o] = sum_b dZ1[b][o], partials per batch chunk:
// part[chunk][o][4] = (dW1[o][0..2], db1[o]).
__device__ void layer1_grad(const Layer1Grad& g, int blk, TileLds& lds) {
  float(*red)[64][IN + 1] = reinterpret_cast<float(*)[64][IN + 1]>(&lds);
  float* xs = reinterpret_cast<float*>(&red[4]);  // the chunk's inputs, read by every column
  const int by = blk / (H / 64);
  const int o = (blk % (H / 64)) * 64 + (threadIdx.x & 63), ph = threadIdx.x >> 6;
  const int64_t b0 = (int64_t)by * CS_ROWS, b1 = min(g.nb, b0 + CS_ROWS);
  for (int e = threadIdx.x; e < (int)(b1 - b0) * IN; e += 256) xs[e] = g.x[b0 * IN + e];
  __syncthreads();
  float s[IN + 1] = {0.0f, 0.0f, 0.0f, 0.0f};
  // rows b0 + ph, b0 + ph + 4, ... accumulated in order; the loads of 32 of them are issued first
  for (int64_t b = b0 + ph; b < b1; b += 128) {
    float d[32];
#pragma unroll
    for (int u = 0; u < 32; ++u) d[u] = b + 4 * u < b1 ? g.dZ[(b + 4 * u) * H + o] : 0.0f;
#pragma unroll
    for (int u = 0; u < 32; ++u) {
      if (b + 4 * u >= b1) break;
      const float* xv = xs + (b + 4 * u - b0) * IN;
#pragma unroll
      for (int i = 0; i < IN; ++i) s[i] = fmaf(d[u], xv[i], s[i]);
      s[IN] += d[u];
    }
  }
#pragma unroll
  for (int i = 0; i <= IN; ++i) red[ph][threadIdx.x & 63][i] = s[i];
  __syncthreads();
  if (ph == 0)
#pragma unroll
    for (int i = 0; i <= IN; ++i)
      g.part[((int64_t)by * H + o) * (IN + 1) + i] =
          red[0][threadIdx.x][i] + red[1][threadIdx.x][i] + red[2][threadIdx.x][i] +
          red[3][threadIdx.x][i];
}

__device__ void reduce_parts(const Reduce& g, int blk) {
  const int e = blk * 256 + threadIdx.x;
  if (e >= g.ne) return;
  float s = 0.0f;
  int z = 0;
  for (; z + 8 <= g.nz; z += 8) {  // added in order; eight loads in flight
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = g.part[(int64_t)(z + u) * g.ne + e];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; z < g.nz; ++z) s += g.part[(int64_t)z * g.ne + e];
  g.out[e] = s;
}

// Jobs of one launch: a column sum first (few blocks, the longest chains), a product, and with
// WGRAD the split-K product of a weight gradient; blocks[i] is the number of blocks of job i.
struct ProductJobs {
  int blocks[3];
  ColSum cs;
  Product p[2];
};
template <int EPI, bool WGRAD>
__global__ __launch_bounds__(256) void products_kernel(ProductJobs j) {
  __shared__ TileLds lds;
  int blk = blockIdx.x;
  if (WGRAD) {
    if (blk < j.blocks[0]) {
      col_sum(j.cs, blk, lds);
      return;
    }
    blk -= j.blocks[0];
  }
  if (!WGRAD || blk < j.blocks[1])
    product<EPI>(j.p[0], blk, lds);
  else
    product<EPI_PART>(j.p[1], blk - j.blocks[1], lds);
}

// The last jobs: first-layer gradient partials and the reductions of all earlier partials.
constexpr int NRED = 6;
struct FinishJobs {
  int blocks[1 + NRED];
  Layer1Grad l1;
  Reduce r[NRED];
  const float* loss_part;  // NULL: no loss
  int n_loss;
  float* loss;
};
__global__ __launch_bounds__(256) void finish_kernel(FinishJobs j) {
  __shared__ TileLds lds;
  int blk = blockIdx.x;
  if (blk < j.blocks[0]) {
    layer1_grad(j.l1, blk, lds);
    return;
  }
  blk -= j.blocks[0];
#pragma unroll
  for (int q = 0; q < NRED; ++q) {
    if (blk < j.blocks[1 + q]) {
      reduce_parts(j.r[q], blk);
      return;
    }
    blk -= j.blocks[1 + q];
  }
  if (!j.loss_part) return;
  float* red = reinterpret_cast<float*>(&lds);
  float s = 0.0f;
  for (int i = threadIdx.x; i < j.n_loss; i += 256) s += j.loss_part[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) j.loss[0] = red[0];
}

__global__ void layer1_grad_finish(const float* __restrict__ part, int nz, float* __restrict__ dW1,
                                   float* __restrict__ db1) {
  const int o = blockIdx.x * blockDim.x + threadIdx.x;
  if (o >= H) return;
  float s[IN + 1] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
  for (int z = 0; z < nz; ++z) {
    const float4 v = *reinterpret_cast<const float4*>(part + ((int64_t)z * H + o) * (IN + 1));
    s[0] += v.x;
    s[1] += v.y;
    s[2] += v.z;
    s[3] += v.w;
  }
#pragma unroll
  for (int i = 0; i < IN; ++i) dW1[o * IN + i] = s[i];
  db1[o] = s[IN];
}

// The matrix-core weights W2, W3, W4 to BF16, W2 and W3 transposed as well, and the first layer:
// Z1[b][o] = sum_i x[b][i] bf16(W1[o][i]) + b1[o], A1 = bf16(silu(Z1)) in both orders (a thread
// takes one neuron and eight points).
constexpr int L1_PTS = 8;
__global__ __launch_bounds__(256) void first_kernel(const float* __restrict__ p,
                                                    const float* __restrict__ x, int64_t nb,
                                                    int wblocks, uint16_t* __restrict__ w2,
                                                    uint16_t* __restrict__ w3,
                                                    uint16_t* __restrict__ w4,
                                                    uint16_t* __restrict__ w2t,
                                                    uint16_t* __restrict__ w3t,
                                                    float* __restrict__ Z,
                                                    uint16_t* __restrict__ A,
                                                    uint16_t* __restrict__ At, int64_t ldt) {
  if ((int)blockIdx.x < wblocks) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < 2 * H * H) {
      const int e = i < H * H ? i : i - H * H;
      const uint16_t h = f2bf(p[(i < H * H ? OW2 : OW3) + e]);
      const int o = e / H, c = e % H;
      (i < H * H ? w2 : w3)[e] = h;
      (i < H * H ? w2t : w3t)[c * H + o] = h;
    } else if (i < 2 * H * H + OUT * H) {
      w4[i - 2 * H * H] = f2bf(p[OW4 + i - 2 * H * H]);
    }
    return;
  }
  const int o = threadIdx.x;
  const int64_t b0 = (int64_t)(blockIdx.x - wblocks) * L1_PTS;
  float w[IN];
#pragma unroll
  for (int i = 0; i < IN; ++i) w[i] = bf2f(f2bf(p[OW1 + o * IN + i]));
  const float bias = p[OB1 + o];
  uint16_t h[L1_PTS];
#pragma unroll
  for (int e = 0; e < L1_PTS; ++e) {
    const int64_t b = b0 + e;
    h[e] = 0;
    if (b >= nb) continue;
    float z = bias;
#pragma unroll
    for (int i = 0; i < IN; ++i) z = fmaf(x[b * IN + i], w[i], z);
    h[e] = f2bf(silu(z));
    Z[b * H + o] = z;
    A[b * H + o] = h[e];
  }
  if (At) {  // ldt is nb rounded up to 8: the padding may be written
    uint4 v;
    memcpy(&v, h, 16);
    *reinterpret_cast<uint4*>(At + (int64_t)o * ldt + b0) = v;
  }
}

// A given output gradient into the workspace: fp32 copy, BF16 in both orders.
__global__ void seed_kernel(const float* __restrict__ dy, int64_t nb, float* __restrict__ dY,
                            uint16_t* __restrict__ dYb, uint16_t* __restrict__ dYt, int64_t ldt) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nb * OUT) return;
  const float d = dy[i];
  const uint16_t h = f2bf(d);
  dY[i] = d;
  dYb[i] = h;
  dYt[(i % OUT) * ldt + i / OUT] = h;
}

__global__ void adam_kernel(float* __restrict__ p, const float* __restrict__ g,
                            float* __restrict__ m, float* __restrict__ v, int64_t n, float lr,
                            float b1, float b2, float eps, float c1, float c2, float wd) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * ((mi / c1) / (sqrtf(vi / c2) + eps) + wd * p[i]);
}

// Packed inference form (layout in ssc_mlp.h).
__global__ void pack_kernel(const float* __restrict__ p, uint16_t* __restrict__ pk16,
                            float* __restrict__ pk32) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 2 * FRAG_L + FRAG_4) {
    int64_t r = i;
    const float* W;
    int rows;
    if (r < FRAG_L) { W = p + OW2; rows = H; }
    else if (r < 2 * FRAG_L) { r -= FRAG_L; W = p + OW3; rows = H; }
    else { r -= 2 * FRAG_L; W = p + OW4; rows = OUT; }
    // fragment order [tile m][k-step j][lane][e] of v_mfma_f32_16x16x32_bf16's A operand
    const int e = (int)(r & 7), l = (int)((r >> 3) & 63);
    const int64_t mj = r >> 9;
    const int j = (int)(mj % (H / 32)), m = (int)(mj / (H / 32));
    const int row = 16 * m + (l & 15);
    const int col = kperm(32 * j + 8 * (l >> 4) + e);
    pk16[i] = row < rows ? f2bf(W[(int64_t)row * H + col]) : (uint16_t)0;
  }
  if (i < PK_F32_END) {
    float v;
    if (i < PK_B1) v = bf2f(f2bf(p[OW1 + i]));
    else if (i < PK_B2) v = p[OB1 + (i - PK_B1)];
    else if (i < PK_B3) v = p[OB2 + (i - PK_B2)];
    else if (i < PK_B4) v = p[OB3 + (i - PK_B3)];
    else v = (i - PK_B4) < OUT ? p[OB4 + (i - PK_B4)] : 0.0f;
    pk32[i] = v;
  }
}

// Packed transposes of the input vector-Jacobian product (layout in ssc_mlp.h).
__global__ void pack_vjp_kernel(const float* __restrict__ p, uint16_t* __restrict__ pkv,
                                float* __restrict__ w4t) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < H * OUT) {  // W4^T [n][o] = W4[o][n], BF16-rounded values in fp32
    const int n = (int)(i / OUT), o = (int)(i % OUT);
    w4t[i] = bf2f(f2bf(p[OW4 + (int64_t)o * H + n]));
  }
  if (i >= PKV_BF16_END) return;
  const int e = (int)(i & 7), l = (int)((i >> 3) & 63);
  int64_t r = i - PKV_W3T;
  const float* W = p + OW3;
  if (r >= FRAG_L) { r -= FRAG_L; W = p + OW2; }
  const int64_t mj = r >> 9;
  const int j = (int)(mj % (H / 32)), m = (int)(mj / (H / 32));
  const int row = 16 * m + (l & 15);                    // input neuron of the layer
  const int col = kperm(32 * j + 8 * (l >> 4) + e);      // output neuron of the layer
  pkv[i] = f2bf(W[(int64_t)col * H + row]);
}

}  // namespace mlp

__global__ __launch_bounds__(256) void mlp_vjp_kernel(const uint16_t* __restrict__ pk16,
                                                      const float* __restrict__ pk32,
                                                      const uint16_t* __restrict__ pkv,
                                                      const float* __restrict__ x,
                                                      const float* __restrict__ dy, int64_t nb,
                                                      float* __restrict__ dx) {
  const int64_t p = ((int64_t)blockIdx.x * 256 + threadIdx.x) / 64 * 16 + (threadIdx.x & 15);
  const bool ok = p < nb;
  const float x0 = ok ? x[3 * p] : 0.0f, x1 = ok ? x[3 * p + 1] : 0.0f, x2 = ok ? x[3 * p + 2] : 0.0f;
  float d[4], yo[4], o[3];
#pragma unroll
  for (int j = 0; j < 4; ++j) d[j] = ok ? dy[4 * p + j] : 0.0f;
  GlobalWeights gw{pk16, pkv};
  mlp_tile_input_vjp(gw, pk32, x0, x1, x2, d, yo, o);
  if (ok && (threadIdx.x & 63) < 16)
#pragma unroll
    for (int j = 0; j < 3; ++j) dx[3 * p + j] = o[j];
}

__global__ __launch_bounds__(256) void mlp_infer_kernel(const uint16_t* __restrict__ pk16,
                                                        const float* __restrict__ pk32,
                                                        const float* __restrict__ x, int64_t nb,
                                                        float* __restrict__ y) {
  const int64_t p = ((int64_t)blockIdx.x * 256 + threadIdx.x) / 64 * 16 + (threadIdx.x & 15);
  const bool ok = p < nb;
  const float x0 = ok ? x[3 * p] : 0.0f, x1 = ok ? x[3 * p + 1] : 0.0f, x2 = ok ? x[3 * p + 2] : 0.0f;
  float o[4];
  GlobalWeights gw{pk16};
  mlp_tile_forward(gw, pk32, x0, x1, x2, o);
  if (ok && (threadIdx.x & 63) < 16)
#pragma unroll
    for (int j = 0; j < 4; ++j) y[4 * p + j] = o[j];
}

// ------------------------------------------------------------------------------------------
// host orchestration
// ------------------------------------------------------------------------------------------
namespace {

using namespace mlp;

struct Workspace {
  float *Z1, *Z2, *Z3, *dZ3, *dZ2, *dZ1, *dY, *loss_part;
  float *pW4, *pW3, *pW2, *pb4, *pb3, *pb2, *pl1;  // partials of the gradient sums
  uint16_t *A1, *A2, *A3, *A1t, *A2t, *A3t, *dZ3b, *dZ2b, *dZ3t, *dZ2t, *dYb, *dYt;
  uint16_t *W2b, *W3b, *W4b, *W2t, *W3t;
  int64_t ldt;  // row pitch of the transposed arrays: the batch rounded up to 8
  int64_t bytes;
};

int64_t splitk_for(int64_t nb) {
  int64_t z = nb / 512;
  return z < 1 ? 1 : (z > 64 ? 64 : z);
}
int64_t chunks_of(int64_t nb) { return (nb + CS_ROWS - 1) / CS_ROWS; }

// Layout of the workspace for a batch; base NULL: the size only.
Workspace carve(void* base, int64_t nb) {
  Workspace w;
  int64_t off = 0;
  base = (void*)(((uintptr_t)base + 63) & ~(uintptr_t)63);
  auto take = [&](int64_t bytes) {
    char* r = base ? (char*)base + off : nullptr;
    off += (bytes + 63) / 64 * 64;
    return r;
  };
  auto f32 = [&](int64_t n) { return (float*)take(n * 4); };
  auto b16 = [&](int64_t n) { return (uint16_t*)take(n * 2); };
  const int64_t nz = splitk_for(nb), nc = chunks_of(nb);
  w.ldt = (nb + 7) / 8 * 8;
  // The backward pass takes no room of its own for a point: a layer's gradient replaces its
  // pre-activations element by element, and its BF16 copies take arrays that the launches before
  // have read for the last time (6.2 KB a point; 10.3 with arrays of their own).
  w.Z1 = f32(nb * H); w.Z2 = f32(nb * H);
  w.Z3 = f32(std::max(nb * H, nz * H * H));
  w.dZ3 = w.Z3; w.dZ2 = w.Z2; w.dZ1 = w.Z1;
  w.dY = f32(nb * OUT);
  w.loss_part = f32((nb + GT - 1) / GT);
  w.pW4 = f32(nz * OUT * H); w.pW3 = f32(nz * H * H);
  w.pW2 = w.Z3;  // formed by the third launch; dZ3 is read by the first two
  w.pb4 = f32(nc * OUT); w.pb3 = f32(nc * H); w.pb2 = f32(nc * H); w.pl1 = f32(nc * H * (IN + 1));
  w.A1 = b16(w.ldt * H); w.A2 = b16(nb * H); w.A3 = b16(nb * H);
  w.A1t = b16(w.ldt * H); w.A2t = b16(w.ldt * H); w.A3t = b16(w.ldt * H);
  w.dZ3b = w.A3; w.dZ3t = w.A1;   // A3 and A1 are read by the forward pass only,
  w.dZ2b = w.A2; w.dZ2t = w.A3t;  // A2 too, A3t by the first backward launch
  w.dYb = b16(nb * OUT); w.dYt = b16(w.ldt * OUT);
  w.W2b = b16(H * H); w.W3b = b16(H * H); w.W4b = b16(OUT * H);
  w.W2t = b16(H * H); w.W3t = b16(H * H);
  w.bytes = off + 64;  // room to align the caller's base
  return w;
}

int64_t ws_bytes(int64_t nb) { return carve(nullptr, nb).bytes; }

inline unsigned nblk(int64_t n, int b = 256) { return (unsigned)((n + b - 1) / b); }

Product make_product(Operand a, Operand b, int K, int nz, int epi) {
  Product g = {};
  g.a = a;
  g.b = b;
  g.K = K;
  g.kchunk = ((K + nz - 1) / nz + GK - 1) / GK * GK;
  g.tm = (int)nblk(a.rows, GT);
  g.tn = (int)nblk(b.rows, GT);
  g.epi = epi;
  return g;
}
int product_blocks(const Product& g) {
  return g.tm * g.tn * ((g.K + g.kchunk - 1) / g.kchunk);
}

void launch_product(const Product& p, hipStream_t st) {
  ProductJobs j = {};
  j.p[0] = p;
  j.blocks[1] = product_blocks(p);
  const dim3 grid((unsigned)j.blocks[1]);
  if (p.epi == EPI_ACT)
    hipLaunchKernelGGL((products_kernel<EPI_ACT, false>), grid, dim3(256), 0, st, j);
  else
    hipLaunchKernelGGL((products_kernel<EPI_OUT, false>), grid, dim3(256), 0, st, j);
}
// One backward launch: bias column sums, the layer below's gradient, the weight gradient.
void launch_backward(const ColSum& cs, const Product& d, const Product& w, hipStream_t st) {
  ProductJobs j = {};
  j.cs = cs;
  j.blocks[0] = (int)(((cs.ncol + 63) / 64) * chunks_of(cs.nb));
  j.p[0] = d;
  j.blocks[1] = product_blocks(d);
  j.p[1] = w;
  j.blocks[2] = product_blocks(w);
  hipLaunchKernelGGL((products_kernel<EPI_DACT, true>),
                     dim3((unsigned)(j.blocks[0] + j.blocks[1] + j.blocks[2])), dim3(256), 0, st, j);
}

// Loss of the training step: targets, weights and their sum (1 / sum, or the sum in device memory).
struct LossArgs {
  const float *target, *weight, *wsum_dev;
  float inv_wsum;
};

// grad: keep the transposed activations for the backward pass; loss: form dY as well.
void forward(const float* p, const float* x, int64_t nb, float* y, Workspace& w, bool grad,
             const LossArgs* loss, hipStream_t st) {
  const unsigned wblocks = nblk(2 * H * H + OUT * H);
  hipLaunchKernelGGL(first_kernel, dim3(wblocks + nblk(nb, L1_PTS)), dim3(256), 0, st, p, x, nb,
                     (int)wblocks, w.W2b, w.W3b, w.W4b, w.W2t, w.W3t, w.Z1, w.A1,
                     grad ? w.A1t : nullptr, w.ldt);
  const uint16_t* Ain[2] = {w.A1, w.A2};
  uint16_t *Aout[2] = {w.A2, w.A3}, *At[2] = {w.A2t, w.A3t};
  const uint16_t* Wb[2] = {w.W2b, w.W3b};
  float* Z[2] = {w.Z2, w.Z3};
  const int64_t ob[2] = {OB2, OB3};
  for (int s = 0; s < 2; ++s) {
    Product g = make_product({Ain[s], H, 1, (int)nb}, {Wb[s], H, 1, H}, H, 1, EPI_ACT);
    g.bias = p + ob[s];
    g.out = Z[s];
    g.out16 = Aout[s];
    g.out16t = grad ? At[s] : nullptr;
    g.ldt = w.ldt;
    launch_product(g, st);
  }
  Product g = make_product({w.A3, H, 1, (int)nb}, {w.W4b, H, 1, OUT}, H, 1, EPI_OUT);
  g.bias = p + OB4;
  g.out = y;
  if (loss) {
    g.target = loss->target;
    g.weight = loss->weight;
    g.wsum_dev = loss->wsum_dev;
    g.inv_wsum = loss->inv_wsum;
    g.dY = w.dY;
    g.out16 = w.dYb;
    g.out16t = w.dYt;
    g.ldt = w.ldt;
    g.loss_part = w.loss_part;
  }
  launch_product(g, st);
}

// Backward from dY (fp32 in w.dY, BF16 in w.dYb and w.dYt) given a forward with the same
// workspace and its transposed activations; loss: also add up the loss partials.
void backward(const float* x, int64_t nb, float* g, Workspace& w, float* loss, hipStream_t st) {
  const int nz = (int)splitk_for(nb), n = (int)nb;
  const int nc = (int)chunks_of(nb);
  // each launch: the gradient of one layer's weights and biases, and the next layer down
  Product w4 = make_product({w.dYt, w.ldt, 1, OUT}, {w.A3t, w.ldt, 1, H}, n, nz, EPI_PART);
  w4.out = w.pW4;
  Product d3 = make_product({w.dYb, OUT, 1, n}, {w.W4b, 1, H, H}, OUT, 1, EPI_DACT);
  d3.Z = w.Z3; d3.out = w.dZ3; d3.out16 = w.dZ3b; d3.out16t = w.dZ3t; d3.ldt = w.ldt;
  const ColSum b4{w.dY, w.pb4, nb, OUT};
  launch_backward(b4, d3, w4, st);

  Product w3 = make_product({w.dZ3t, w.ldt, 1, H}, {w.A2t, w.ldt, 1, H}, n, nz, EPI_PART);
  w3.out = w.pW3;
  Product d2 = make_product({w.dZ3b, H, 1, n}, {w.W3t, H, 1, H}, H, 1, EPI_DACT);
  d2.Z = w.Z2; d2.out = w.dZ2; d2.out16 = w.dZ2b; d2.out16t = w.dZ2t; d2.ldt = w.ldt;
  const ColSum b3{w.dZ3, w.pb3, nb, H};
  launch_backward(b3, d2, w3, st);

  Product w2 = make_product({w.dZ2t, w.ldt, 1, H}, {w.A1t, w.ldt, 1, H}, n, nz, EPI_PART);
  w2.out = w.pW2;
  Product d1 = make_product({w.dZ2b, H, 1, n}, {w.W2t, H, 1, H}, H, 1, EPI_DACT);
  d1.Z = w.Z1; d1.out = w.dZ1;
  const ColSum b2{w.dZ2, w.pb2, nb, H};
  launch_backward(b2, d1, w2, st);

  FinishJobs f = {};
  f.l1 = Layer1Grad{w.dZ1, x, w.pl1, nb};
  f.blocks[0] = (H / 64) * nc;
  const int z = (n + w3.kchunk - 1) / w3.kchunk;  // chunks written by the weight products
  const Reduce r[NRED] = {{w.pW3, g + OW3, z, H * H}, {w.pW2, g + OW2, z, H * H},
                          {w.pW4, g + OW4, z, OUT * H}, {w.pb4, g + OB4, nc, OUT},
                          {w.pb3, g + OB3, nc, H}, {w.pb2, g + OB2, nc, H}};
  unsigned total = f.blocks[0];
  for (int q = 0; q < NRED; ++q) {
    f.r[q] = r[q];
    f.blocks[1 + q] = (int)nblk(r[q].ne);
    total += f.blocks[1 + q];
  }
  if (loss) {
    f.loss_part = w.loss_part;
    f.n_loss = (int)nblk(nb, GT);
    f.loss = loss;
    ++total;
  }
  hipLaunchKernelGGL(finish_kernel, dim3(total), dim3(256), 0, st, f);
  hipLaunchKernelGGL(layer1_grad_finish, dim3(1), dim3(H), 0, st, w.pl1, nc, g + OW1, g + OB1);
}

}  // namespace
}  // namespace ssc

using namespace ssc;
using namespace ssc::mlp;

extern "C" {

int64_t ssc_mlp_num_params(void) { return NPARAM; }

int64_t ssc_mlp_packed_bytes(void) { return PACKED_BYTES; }

int64_t ssc_mlp_workspace_bytes(int64_t batch) { return batch > 0 ? ws_bytes(batch) : 0; }

int ssc_mlp_forward(const float* params, const float* x, int64_t batch, float* y, void* workspace,
                    int64_t workspace_bytes, void* stream) {
  if (!params || !x || !y || !workspace || batch <= 0)
    return fail(SSC_E_ARG, "ssc_mlp_forward: NULL pointer or empty batch");
  if (batch > (1 << 24)) return fail(SSC_E_LIMIT, "ssc_mlp_forward: batch above 16M");
  if (workspace_bytes < ws_bytes(batch)) return fail(SSC_E_ARG, "ssc_mlp_forward: workspace too small");
  Workspace w = carve(workspace, batch);
  forward(params, x, batch, y, w, false, nullptr, (hipStream_t)stream);
  return check_launch("ssc_mlp_forward");
}

static int loss_backward(const char* name, const float* params, const float* x,
                         const float* target, const float* weight, float weight_sum,
                         const float* weight_sum_dev, int64_t batch, float* y, float* grads,
                         float* loss, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!params || !x || !target || !y || !grads || !loss || !workspace || batch <= 0)
    return fail(SSC_E_ARG, std::string(name) + ": NULL pointer or empty batch");
  if (batch > (1 << 24)) return fail(SSC_E_LIMIT, std::string(name) + ": batch above 16M");
  if (workspace_bytes < ws_bytes(batch))
    return fail(SSC_E_ARG, std::string(name) + ": workspace too small");
  if (!weight_sum_dev && !(weight_sum > 0.0f))
    return fail(SSC_E_ARG, std::string(name) + ": weight_sum must be > 0");
  hipStream_t st = (hipStream_t)stream;
  Workspace w = carve(workspace, batch);
  const LossArgs la{target, weight, weight_sum_dev, weight_sum_dev ? 0.0f : 1.0f / weight_sum};
  forward(params, x, batch, y, w, true, &la, st);
  backward(x, batch, grads, w, loss, st);
  return check_launch(name);
}

int ssc_mlp_loss_backward(const float* params, const float* x, const float* target,
                          const float* weight, float weight_sum, int64_t batch, float* y,
                          float* grads, float* loss, void* workspace, int64_t workspace_bytes,
                          void* stream) {
  return loss_backward("ssc_mlp_loss_backward", params, x, target, weight, weight_sum, nullptr,
                       batch, y, grads, loss, workspace, workspace_bytes, stream);
}

int ssc_mlp_loss_backward_dev(const float* params, const float* x, const float* target,
                              const float* weight, const float* weight_sum, int64_t batch,
                              float* y, float* grads, float* loss, void* workspace,
                              int64_t workspace_bytes, void* stream) {
  if (!weight_sum) return fail(SSC_E_ARG, "ssc_mlp_loss_backward_dev: NULL weight_sum");
  return loss_backward("ssc_mlp_loss_backward_dev", params, x, target, weight, 0.0f,
                       weight_sum, batch, y, grads, loss, workspace, workspace_bytes, stream);
}

int ssc_mlp_backward(const float* params, const float* x, const float* dy, int64_t batch,
                     float* grads, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!params || !x || !dy || !grads || !workspace || batch <= 0)
    return fail(SSC_E_ARG, "ssc_mlp_backward: NULL pointer or empty batch");
  if (workspace_bytes < ws_bytes(batch)) return fail(SSC_E_ARG, "ssc_mlp_backward: workspace too small");
  hipStream_t st = (hipStream_t)stream;
  Workspace w = carve(workspace, batch);
  // recompute the forward into the workspace; dy takes the place of the loss gradient (and of the
  // outputs, which are not asked for)
  forward(params, x, batch, w.dY, w, true, nullptr, st);
  hipLaunchKernelGGL(seed_kernel, dim3(nblk(batch * OUT)), dim3(256), 0, st, dy, batch, w.dY, w.dYb,
                     w.dYt, w.ldt);
  backward(x, batch, grads, w, nullptr, st);
  return check_launch("ssc_mlp_backward");
}

int ssc_mlp_adam(float* params, const float* grads, float* m, float* v, int64_t n, float lr,
                 float beta1, float beta2, float eps, int32_t step, float weight_decay,
                 void* stream) {
  if (!params || !grads || !m || !v || n <= 0 || step <= 0)
    return fail(SSC_E_ARG, "ssc_mlp_adam: bad argument");
  const float c1 = 1.0f - powf(beta1, (float)step), c2 = 1.0f - powf(beta2, (float)step);
  hipLaunchKernelGGL(adam_kernel, dim3(nblk(n)), dim3(256), 0, (hipStream_t)stream, params, grads,
                     m, v, n, lr, beta1, beta2, eps, c1, c2, weight_decay);
  return check_launch("ssc_mlp_adam");
}

int ssc_mlp_pack(const float* params, void* packed, void* stream) {
  if (!params || !packed) return fail(SSC_E_ARG, "ssc_mlp_pack: NULL pointer");
  uint16_t* pk16 = (uint16_t*)packed;
  float* pk32 = (float*)((char*)packed + PK_F32_BASE_BYTES);
  hipLaunchKernelGGL(pack_kernel, dim3(nblk(2 * FRAG_L + FRAG_4)), dim3(256), 0, (hipStream_t)stream,
                     params, pk16, pk32);
  return check_launch("ssc_mlp_pack");
}

int64_t ssc_mlp_packed_vjp_bytes(void) { return PACKED_VJP_BYTES; }

int ssc_mlp_pack_vjp(const float* params, void* packed_vjp, void* stream) {
  if (!params || !packed_vjp) return fail(SSC_E_ARG, "ssc_mlp_pack_vjp: NULL pointer");
  hipLaunchKernelGGL(pack_vjp_kernel, dim3(nblk(PKV_BF16_END)), dim3(256), 0, (hipStream_t)stream,
                     params, (uint16_t*)packed_vjp, (float*)((char*)packed_vjp + PKV_W4T_BYTES));
  return check_launch("ssc_mlp_pack_vjp");
}

int ssc_mlp_input_vjp(const void* packed, const void* packed_vjp, const float* x, const float* dy,
                      int64_t batch, float* dx, void* stream) {
  if (!packed || !packed_vjp || !x || !dy || !dx || batch < 0)
    return fail(SSC_E_ARG, "ssc_mlp_input_vjp: bad argument");
  if (batch == 0) return SSC_OK;
  const uint16_t* pk16 = (const uint16_t*)packed;
  const float* pk32 = (const float*)((const char*)packed + PK_F32_BASE_BYTES);
  const int64_t blocks = (batch + 63) / 64;  // 4 waves x 16 points
  hipLaunchKernelGGL(mlp_vjp_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                     pk16, pk32, (const uint16_t*)packed_vjp, x, dy, batch, dx);
  return check_launch("ssc_mlp_input_vjp");
}

int ssc_mlp_infer(const void* packed, const float* x, int64_t batch, float* y, void* stream) {
  if (!packed || !x || !y || batch < 0) return fail(SSC_E_ARG, "ssc_mlp_infer: bad argument");
  if (batch == 0) return SSC_OK;
  const uint16_t* pk16 = (const uint16_t*)packed;
  const float* pk32 = (const float*)((const char*)packed + PK_F32_BASE_BYTES);
  const int64_t blocks = (batch + 63) / 64;  // 4 waves x 16 points
  hipLaunchKernelGGL(mlp_infer_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                     pk16, pk32, x, batch, y);
  return check_launch("ssc_mlp_infer");
}

}  // extern "C"
