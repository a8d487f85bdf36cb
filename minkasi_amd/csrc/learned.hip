// Learned map-space preconditioner: linear dilated 3x3 convolutions.
//
// The preconditioner is M = S (alpha I + K^T K) S with S = diag(sqrt(1/hits))
// (zero on unhit pixels) and K a chain of linear 3x3 convolutions (no
// activations), so M is symmetric positive semidefinite by construction and
// positive definite on hit pixels when alpha > 0.  Layer l has dilation
// dil_l: tap d = 3*di + dj reads offset (dil*(di-1), dil*(dj-1)).
//
//   conv3x3: y[b,o,p] (+)= sum_{c,d} w[o,c,d] x[b,c,p+off_d]   (zero padding)
//            The adjoint layer is the same kernel with the weights
//            transposed in (o,c) and flipped in d (mk_conv3x3_adjoint_weights).
//   wgrad:   g[o,c,d] = sum_{b,p} a[b,o,p] x[b,c,p+off_d]
//            the weight gradient of a forward layer (a = output gradient,
//            x = layer input) and of an adjoint layer (a = layer input,
//            x = output gradient).
//
// A level network outside training needs no activations: its M r runs on
// composed 5x5 stencils, one pass per level (mk_precon_levels_f32, below).
//
// Tiling is polyphase: a workgroup owns the 16x16 lattice of pixels
// (i0 + dil*a, j0 + dil*c) inside a 16*dil square super-tile, so a dilated
// tap is a +-1 lattice step and the LDS tile is 18x18 per channel whatever
// the dilation.  Activations are planar FP32 [B][C][H][W]; arithmetic is FP32
// with the weights read through uniform (scalar) loads.  wgrad reduces fixed
// per-workgroup partials in a fixed order, so every result is deterministic.
#include "common.h"

namespace {

constexpr int TS = 16;            // lattice tile side
constexpr int HS = TS + 2;        // with the +-1 halo
constexpr int XP = HS + 1;        // LDS row pitch of an input tile
constexpr int XCH = HS * XP;      // LDS channel stride of an input tile (342)
constexpr int AP = TS + 1;        // LDS row pitch of an output-gradient tile
constexpr int ACH = TS * AP + 1;  // LDS channel stride of an output-gradient tile (273)
constexpr int MAXC = 16;
constexpr int kWgradGroups = 2048;

struct Tiling {
  int H, W, dil, ntj, per_img;  // per_img = ntiles_i * ntiles_j * dil^2
  __device__ void locate(int bid, int& b, int& i0, int& j0) const {
    b = bid / per_img;
    int rem = bid - b * per_img;
    int d2 = dil * dil;
    int T = rem / d2, ph = rem - T * d2;
    int ti = T / ntj, tj = T - ti * ntj;
    i0 = ti * TS * dil + ph / dil;
    j0 = tj * TS * dil + ph % dil;
  }
};

inline Tiling make_tiling(int H, int W, int dil) {
  Tiling t;
  t.H = H; t.W = W; t.dil = dil;
  int nti = (int)mk::cdiv(H, (int64_t)TS * dil);
  t.ntj = (int)mk::cdiv(W, (int64_t)TS * dil);
  t.per_img = nti * t.ntj * dil * dil;
  return t;
}

// Stages channels [0, C) of the lattice tile with halo into LDS (zero outside
// the image).
__device__ inline void stage_halo(float* xs, const float* __restrict__ xb, int C, const Tiling& t, int i0,
                                  int j0) {
  const int64_t plane = (int64_t)t.H * t.W;
  for (int k = threadIdx.x; k < C * HS * HS; k += 256) {
    int c = k / (HS * HS), rq = k - c * (HS * HS);
    int r = rq / HS, q = rq - r * HS;
    int gi = i0 + t.dil * (r - 1), gj = j0 + t.dil * (q - 1);
    float v = 0.f;
    if (gi >= 0 && gi < t.H && gj >= 0 && gj < t.W) v = xb[c * plane + (int64_t)gi * t.W + gj];
    xs[c * XCH + r * XP + q] = v;
  }
}

template <int CIN, int COUT>
__global__ void __launch_bounds__(256) conv3x3_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                      float* __restrict__ y, Tiling t, int accumulate) {
  __shared__ float xs[CIN * XCH];
  int b, i0, j0;
  t.locate(blockIdx.x, b, i0, j0);
  const int64_t plane = (int64_t)t.H * t.W;
  stage_halo(xs, x + (int64_t)b * CIN * plane, CIN, t, i0, j0);
  __syncthreads();
  const int li = threadIdx.x / TS, lj = threadIdx.x % TS;
  float acc[COUT];
#pragma unroll
  for (int o = 0; o < COUT; o++) acc[o] = 0.f;
#pragma unroll 1
  for (int c = 0; c < CIN; c++) {
    float v[9];
#pragma unroll
    for (int d = 0; d < 9; d++) v[d] = xs[c * XCH + (li + d / 3) * XP + lj + d % 3];
#pragma unroll
    for (int o = 0; o < COUT; o++) {
      const float* wo = w + (o * CIN + c) * 9;
#pragma unroll
      for (int d = 0; d < 9; d++) acc[o] = fmaf(wo[d], v[d], acc[o]);
    }
  }
  const int gi = i0 + t.dil * li, gj = j0 + t.dil * lj;
  if (gi < t.H && gj < t.W) {
    float* yb = y + (int64_t)b * COUT * plane + (int64_t)gi * t.W + gj;
#pragma unroll
    for (int o = 0; o < COUT; o++) {
      float v = acc[o];
      if (accumulate) v += yb[o * plane];
      yb[o * plane] = v;
    }
  }
}

// Thread k < CO*CI owns weights (o, c) = (k / CI, k % CI) and keeps their 9
// taps in registers over every tile the workgroup visits; the 3x3 input
// window slides along each lattice row.
template <int CO, int CI>
__global__ void __launch_bounds__(256) wgrad_kernel(const float* __restrict__ a, const float* __restrict__ x,
                                                    Tiling t, int total, float* __restrict__ part) {
  __shared__ float as[CO * ACH];
  __shared__ float xs[CI * XCH];
  const int64_t plane = (int64_t)t.H * t.W;
  const int k = threadIdx.x;
  const bool active = k < CO * CI;
  const int o = active ? k / CI : 0, c = active ? k % CI : 0;
  float g[9];
#pragma unroll
  for (int d = 0; d < 9; d++) g[d] = 0.f;
  for (int bid = blockIdx.x; bid < total; bid += gridDim.x) {
    int b, i0, j0;
    t.locate(bid, b, i0, j0);
    const float* ab = a + (int64_t)b * CO * plane;
    for (int e = threadIdx.x; e < CO * TS * TS; e += 256) {
      int oo = e / (TS * TS), rq = e - oo * (TS * TS);
      int r = rq / TS, q = rq - r * TS;
      int gi = i0 + t.dil * r, gj = j0 + t.dil * q;
      float v = 0.f;
      if (gi < t.H && gj < t.W) v = ab[oo * plane + (int64_t)gi * t.W + gj];
      as[oo * ACH + r * AP + q] = v;
    }
    stage_halo(xs, x + (int64_t)b * CI * plane, CI, t, i0, j0);
    __syncthreads();
    if (active) {
      const float* ao = as + o * ACH;
      const float* xc = xs + c * XCH;
#pragma unroll 1
      for (int r = 0; r < TS; r++) {
        float w0[3], w1[3], w2[3];  // window columns q-1+{0,1,2} (halo coordinates q, q+1, q+2)
#pragma unroll
        for (int di = 0; di < 3; di++) {
          w0[di] = xc[(r + di) * XP + 0];
          w1[di] = xc[(r + di) * XP + 1];
        }
#pragma unroll 4
        for (int q = 0; q < TS; q++) {
#pragma unroll
          for (int di = 0; di < 3; di++) w2[di] = xc[(r + di) * XP + q + 2];
          const float av = ao[r * AP + q];
#pragma unroll
          for (int di = 0; di < 3; di++) {
            g[3 * di + 0] = fmaf(av, w0[di], g[3 * di + 0]);
            g[3 * di + 1] = fmaf(av, w1[di], g[3 * di + 1]);
            g[3 * di + 2] = fmaf(av, w2[di], g[3 * di + 2]);
          }
#pragma unroll
          for (int di = 0; di < 3; di++) {
            w0[di] = w1[di];
            w1[di] = w2[di];
          }
        }
      }
    }
    __syncthreads();
  }
  if (active) {
    float* out = part + (int64_t)blockIdx.x * (CO * CI * 9) + (o * CI + c) * 9;
#pragma unroll
    for (int d = 0; d < 9; d++) out[d] = g[d];
  }
}

__global__ void __launch_bounds__(256) wgrad_reduce_kernel(const float* __restrict__ part, int nparts, int nw,
                                                           float* __restrict__ g, int accumulate) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nw) return;
  double s = 0.0;  // fixed order; FP64 sum of the FP32 partials
  for (int p = 0; p < nparts; p++) s += (double)part[(int64_t)p * nw + k];
  g[k] = accumulate ? (float)((double)g[k] + s) : (float)s;
}

__global__ void adjoint_weights_kernel(const float* __restrict__ w, int Co, int Ci, float* __restrict__ wt) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= Co * Ci * 9) return;
  int o = k / (Ci * 9), c = (k / 9) % Ci, d = k % 9;
  wt[(c * Co + o) * 9 + (8 - d)] = w[k];
}

// z = s * (exp(log_alpha) * u + g)   (g may be NULL)
__global__ void __launch_bounds__(256) precon_finish_kernel(float* __restrict__ z, const float* __restrict__ s,
                                                            const float* __restrict__ log_alpha,
                                                            const float* __restrict__ u, const float* __restrict__ g,
                                                            int64_t n) {
  const float alpha = expf(log_alpha[0]);
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    float v = alpha * u[i];
    if (g) v += g[i];
    z[i] = s[i] * v;
  }
}

constexpr int kLossGroups = 1024;

__device__ inline double block_sum256(double v, double* sh) {
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
    __syncthreads();
  }
  double out = sh[0];
  __syncthreads();
  return out;
}

// Loss L = sum m * (s*(alpha u + g) - e)^2; q = dL/d(alpha u + g) = 2 m s delta;
// partials of L and of dL/dalpha = sum q u.
__global__ void __launch_bounds__(256) precon_loss_stage1(const float* __restrict__ g, const float* __restrict__ u,
                                                          const float* __restrict__ s, const float* __restrict__ e,
                                                          const float* __restrict__ m,
                                                          const float* __restrict__ log_alpha, int64_t n,
                                                          float* __restrict__ q, double* __restrict__ part) {
  __shared__ double sh[256];
  const float alpha = expf(log_alpha[0]);
  double sl = 0.0, sa = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)kLossGroups * 256) {
    float ui = u[i], si = s[i], mi = m[i];
    float del = si * fmaf(alpha, ui, g[i]) - e[i];
    float qi = 2.f * mi * si * del;
    q[i] = qi;
    sl += (double)mi * (double)del * (double)del;
    sa += (double)qi * (double)ui;
  }
  sl = block_sum256(sl, sh);
  sa = block_sum256(sa, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = sl;
    part[kLossGroups + blockIdx.x] = sa;
  }
}

__global__ void __launch_bounds__(256) precon_loss_stage2(const double* __restrict__ part, double* __restrict__ sc) {
  __shared__ double sh[256];
  double a = 0.0, b = 0.0;
  for (int i = threadIdx.x; i < kLossGroups; i += 256) {
    a += part[i];
    b += part[kLossGroups + i];
  }
  a = block_sum256(a, sh);
  b = block_sum256(b, sh);
  if (threadIdx.x == 0) {
    sc[0] = a;
    sc[1] = b;
  }
}

// Energy-norm loss of one preconditioned step: with z = M r and Az = A z,
// L = (z - e).(Az - r) = ||z - e||_A^2 (A e = r), q = dL/dt = 2 s (Az - r)
// for z = s t, and dL/dalpha = sum q u.
__global__ void __launch_bounds__(256) precon_aloss_stage1(const float* __restrict__ z, const float* __restrict__ az,
                                                           const float* __restrict__ r, const float* __restrict__ e,
                                                           const float* __restrict__ s, const float* __restrict__ u,
                                                           int64_t n, float* __restrict__ q,
                                                           double* __restrict__ part) {
  __shared__ double sh[256];
  double sl = 0.0, sa = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)kLossGroups * 256) {
    double res = (double)az[i] - (double)r[i];
    float qi = (float)(2.0 * (double)s[i] * res);
    q[i] = qi;
    sl += ((double)z[i] - (double)e[i]) * res;
    sa += (double)qi * (double)u[i];
  }
  sl = block_sum256(sl, sh);
  sa = block_sum256(sa, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = sl;
    part[kLossGroups + blockIdx.x] = sa;
  }
}

// Box restriction by f (stride f): y[b,I,J] = f^-2 sum_{a,c<f} x[b, fI+a, fJ+c],
// zero beyond the fine grid; the coarse grid is ceil(H/f) x ceil(W/f).
__global__ void __launch_bounds__(256) restrict_kernel(const float* __restrict__ x, int H, int W, int f, int Hc,
                                                       int Wc, int64_t total, float* __restrict__ y) {
  const float inv = 1.f / (float)(f * f);
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < total; k += (int64_t)gridDim.x * blockDim.x) {
    int64_t b = k / ((int64_t)Hc * Wc);
    int rem = (int)(k - b * Hc * Wc);
    int I = rem / Wc, J = rem - I * Wc;
    const float* xb = x + b * (int64_t)H * W;
    float s = 0.f;
    for (int a = 0; a < f; a++) {
      int i = I * f + a;
      if (i >= H) break;
      for (int c = 0; c < f; c++) {
        int j = J * f + c;
        if (j < W) s += xb[(int64_t)i * W + j];
      }
    }
    y[k] = s * inv;
  }
}

// Adjoint of restrict_kernel: x[b,i,j] (+)= f^-2 y[b, i/f, j/f].
__global__ void __launch_bounds__(256) prolong_kernel(const float* __restrict__ y, int Hc, int Wc, int f, int H, int W,
                                                      int64_t total, float* __restrict__ x, int accumulate) {
  const float inv = 1.f / (float)(f * f);
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < total; k += (int64_t)gridDim.x * blockDim.x) {
    int64_t b = k / ((int64_t)H * W);
    int rem = (int)(k - b * H * W);
    int i = rem / W, j = rem - i * W;
    float v = y[b * (int64_t)Hc * Wc + (int64_t)(i / f) * Wc + j / f] * inv;
    x[k] = accumulate ? x[k] + v : v;
  }
}

// Full-weighting (tent) restriction by f: coarse point I is centred on fine
// position f I + (f-1)/2 and fine pixel i weighs max(0, 2f - |d|) / (2 f^2),
// d = 2i - (2 f I + f - 1), per axis (the weights of a coarse point sum to
// 1 in the interior).  Its adjoint is bilinear interpolation, so coarse
// corrections come back smooth instead of blocky.
__device__ __forceinline__ float tent_w(int i, int I, int f) {
  int d = 2 * i - (2 * f * I + f - 1);
  d = d < 0 ? -d : d;
  return d < 2 * f ? (float)(2 * f - d) : 0.f;
}

__global__ void __launch_bounds__(256) restrict_tent_kernel(const float* __restrict__ x, int H, int W, int f, int Hc,
                                                            int Wc, int64_t total, float* __restrict__ y) {
  const float norm = 1.f / (4.f * (float)f * (float)f * (float)f * (float)f);
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < total; k += (int64_t)gridDim.x * blockDim.x) {
    int64_t b = k / ((int64_t)Hc * Wc);
    int rem = (int)(k - b * Hc * Wc);
    int I = rem / Wc, J = rem - I * Wc;
    const float* xb = x + b * (int64_t)H * W;
    const int i0 = max(0, f * I - f / 2 - 1), i1 = min(H - 1, f * I + f + f / 2);
    const int j0 = max(0, f * J - f / 2 - 1), j1 = min(W - 1, f * J + f + f / 2);
    float s = 0.f;
    for (int i = i0; i <= i1; i++) {
      const float wi = tent_w(i, I, f);
      if (wi == 0.f) continue;
      float r = 0.f;
      for (int j = j0; j <= j1; j++) r = fmaf(tent_w(j, J, f), xb[(int64_t)i * W + j], r);
      s = fmaf(wi, r, s);
    }
    y[k] = s * norm;
  }
}

__global__ void __launch_bounds__(256) prolong_tent_kernel(const float* __restrict__ y, int Hc, int Wc, int f, int H,
                                                           int W, int64_t total, float* __restrict__ x,
                                                           int accumulate) {
  const float norm = 1.f / (4.f * (float)f * (float)f * (float)f * (float)f);
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < total; k += (int64_t)gridDim.x * blockDim.x) {
    int64_t b = k / ((int64_t)H * W);
    int rem = (int)(k - b * H * W);
    int i = rem / W, j = rem - i * W;
    const float* yb = y + b * (int64_t)Hc * Wc;
    // coarse points whose support holds i: I with |2i - (2fI + f - 1)| < 2f
    const int Ilo = max(0, (2 * i - 3 * f + 1) / (2 * f) - 1), Ihi = min(Hc - 1, (2 * i + f + 1) / (2 * f) + 1);
    const int Jlo = max(0, (2 * j - 3 * f + 1) / (2 * f) - 1), Jhi = min(Wc - 1, (2 * j + f + 1) / (2 * f) + 1);
    float v = 0.f;
    for (int I = Ilo; I <= Ihi; I++) {
      const float wi = tent_w(i, I, f);
      if (wi == 0.f) continue;
      for (int J = Jlo; J <= Jhi; J++) v = fmaf(wi * tent_w(j, J, f), yb[(int64_t)I * Wc + J], v);
    }
    v *= norm;
    x[k] = accumulate ? x[k] + v : v;
  }
}

// ---- M r of the level networks in one pass per level ----------------------
//
// K^T K of a level network is, per level, the composition of a 1 -> 16 layer
// and its adjoint.  Written out, it is one 5x5 stencil of the level's map:
//   g[p] = sum_d in(p - off_d) sum_e M[d][e] u[p - off_d + off_e],
//   M[d][e] = sum_o w[o][d] w[o][e],
// whose taps with equal e - d add up to 25 coefficients.  The 16 channels are
// zero outside the image, so on the outermost ring of pixels the terms d that
// leave the image drop out: the ring has its own coefficients, one set per
// combination of edges the pixel touches.
constexpr int kEdge = 4;                       // bit 0: first row/column, bit 1: last
constexpr int kStencil = kEdge * kEdge * 25;   // floats per level: [row edge][column edge][25]

// One workgroup per level: the Gram of the taps and the sums in FP64, rounded
// once (the layers themselves round after every tap and channel).
__global__ void __launch_bounds__(256) level_stencil_kernel(const float* __restrict__ w, float* __restrict__ st) {
  __shared__ double M[81];
  w += (int64_t)blockIdx.x * MAXC * 9;
  st += (int64_t)blockIdx.x * kStencil;
  const int t = threadIdx.x;
  if (t < 81) {
    double m = 0.0;
    for (int o = 0; o < MAXC; o++) m = fma((double)w[o * 9 + t / 9], (double)w[o * 9 + t % 9], m);
    M[t] = m;
  }
  __syncthreads();
  for (int k = t; k < kStencil; k += 256) {
    const int cls = k / 25, tap = k % 25, ce = cls / kEdge, cf = cls % kEdge;
    const int di = tap / 5 - 2, dj = tap % 5 - 2;  // e - d
    double v = 0.0;
    for (int d = 0; d < 9; d++) {
      const int r = d / 3, c = d % 3, er = r + di, ec = c + dj;
      if (er < 0 || er > 2 || ec < 0 || ec > 2) continue;
      if ((r == 2 && (ce & 1)) || (r == 0 && (ce & 2)) || (c == 2 && (cf & 1)) || (c == 0 && (cf & 2))) continue;
      v += M[d * 9 + er * 3 + ec];
    }
    st[k] = (float)v;
  }
}

__device__ __forceinline__ int edge_class(int i, int n) { return (i == 0 ? 1 : 0) | (i == n - 1 ? 2 : 0); }

// Weight of fine index i in coarse index I (per axis) and its norm.
template <bool TENT>
__device__ __forceinline__ float axis_w(int i, int I, int f) {
  if constexpr (TENT) return tent_w(i, I, f);
  return (i >= I * f && i < (I + 1) * f) ? 1.f : 0.f;
}
template <bool TENT>
__device__ __forceinline__ float axis_norm(int f) {
  return TENT ? 1.f / (4.f * (float)f * (float)f * (float)f * (float)f) : 1.f / (float)(f * f);
}

// Restriction of x (times s, where given) by f.  Bandwidth-bound on its input:
// every thread walks down one fine column, adds each sample to the (at most
// two) coarse rows it belongs to, and the workgroup sums each row of column
// sums along the other axis from LDS, so a sample is read 1 + 1/kRC times
// instead of 4 (tent weights reach 2f samples per axis), always along rows.
// 2048^2 by 4, with s: 14 us from 22 + 8 (one thread per coarse sample, and
// the product in a pass of its own).
constexpr int kRC = 4;   // coarse rows per workgroup
constexpr int kRB = 10;  // fine rows loaded at a time

template <bool TENT, bool MUL>
__global__ void __launch_bounds__(256) level_restrict_kernel(const float* __restrict__ x, const float* __restrict__ s,
                                                             int H, int W, int f, int Hc, int Wc, int nbj, int per_img,
                                                             float* __restrict__ y) {
  __shared__ float col[kRC][256 + 1];
  const int b = blockIdx.x / per_img, rem = blockIdx.x - b * per_img;
  const int I0 = (rem / nbj) * kRC, cj = TENT ? 256 / f - 1 : 256 / f, J0 = (rem % nbj) * cj;
  const int jb = f * J0 - (TENT ? f / 2 : 0), j = jb + (int)threadIdx.x;
  const int i0 = f * I0 - (TENT ? f / 2 : 0), ni = TENT ? f * kRC + f : f * kRC;
  float acc[kRC];
#pragma unroll
  for (int k = 0; k < kRC; k++) acc[k] = 0.f;
  if (j >= 0 && j < W) {
    const float* xb = x + (int64_t)b * H * W + j;
    const float* sb = MUL ? s + (int64_t)b * H * W + j : nullptr;
    const int ia = max(i0, 0), ie = min(i0 + ni, H);
    for (int i = ia; i < ie; i += kRB) {  // kRB rows in flight
      float v[kRB];
#pragma unroll
      for (int q = 0; q < kRB; q++) v[q] = i + q < ie ? xb[(int64_t)(i + q) * W] : 0.f;
      if constexpr (MUL) {
        float sv[kRB];
#pragma unroll
        for (int q = 0; q < kRB; q++) sv[q] = i + q < ie ? sb[(int64_t)(i + q) * W] : 0.f;
#pragma unroll
        for (int q = 0; q < kRB; q++) v[q] *= sv[q];
      }
#pragma unroll
      for (int q = 0; q < kRB; q++)
#pragma unroll
        for (int k = 0; k < kRC; k++) {
          const float w = axis_w<TENT>(i + q, I0 + k, f);
          if (w != 0.f) acc[k] = fmaf(w, v[q], acc[k]);  // an infinity stays in the rows that hold it
        }
    }
  }
#pragma unroll
  for (int k = 0; k < kRC; k++) col[k][threadIdx.x] = acc[k];
  __syncthreads();
  const float norm = axis_norm<TENT>(f);
  for (int o = threadIdx.x; o < kRC * cj; o += 256) {
    const int k = o / cj, q = o - k * cj, I = I0 + k, J = J0 + q;
    if (I >= Hc || J >= Wc) continue;
    const int t0 = f * q, nt = TENT ? 2 * f : f;  // fine columns jb + t0 ... of coarse column J
    float v = 0.f;
    for (int t = t0; t < t0 + nt; t++) v = fmaf(axis_w<TENT>(jb + t, J, f), col[k][t], v);
    y[((int64_t)b * Hc + I) * Wc + J] = v * norm;
  }
}

// One level: out = stencil(u) + R^T g, with g the finished next coarser level
// (absent at the coarsest).  FINE: u = s r is formed while the tile is staged
// and out = s (alpha u + stencil(u) + R^T g) is the whole result.  A workgroup
// of 4 waves owns 64 x (4 RPT) pixels with a halo of 2 in LDS; a lane owns one
// column of RPT pixels and slides the 5 values of each row under all the
// outputs they reach, so a pixel takes 5 (1 + 4/RPT) LDS reads and 25 fused
// multiply-adds, with the coefficients in scalar registers.  RPT 8 where that
// still leaves two workgroups per CU, 2 on the smaller levels.  The finest
// level of 2048^2 with its tent prolongation: 22 us (50 MB of traffic) from
// 317 (layer and adjoint over 16 channel planes 256, prolongation 43, product
// and finish 17).
template <bool FINE, bool TENT, int RPT>
__global__ void __launch_bounds__(256) level_kernel(const float* __restrict__ x, const float* __restrict__ s,
                                                    const float* __restrict__ log_alpha,
                                                    const float* __restrict__ st, const float* __restrict__ g, int H,
                                                    int W, int f, int Hc, int Wc, int nbj, int per_img,
                                                    float* __restrict__ out) {
  constexpr int TR = 4 * RPT, LW = 64 + 4, LR = TR + 4;
  __shared__ float us[LR * LW], ring[kStencil];
  const int b = blockIdx.x / per_img, rem = blockIdx.x - b * per_img;
  const int i0 = (rem / nbj) * TR, j0 = (rem % nbj) * 64;
  const bool edge = i0 == 0 || j0 == 0 || i0 + TR >= H || j0 + 64 >= W;
  if (edge)
    for (int k = threadIdx.x; k < kStencil; k += 256) ring[k] = st[k];
  const float* xb = x + (int64_t)b * H * W;
  const float* sb = FINE ? s + (int64_t)b * H * W : nullptr;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  {  // wave w stages rows w, w + 4, ...: 64 columns a row, then the last 4 of all rows at once
    const int gj = j0 + lane - 2;
    float v[LR / 4], sv[LR / 4];
#pragma unroll
    for (int q = 0; q < LR / 4; q++) {
      const int gi = i0 + wave + 4 * q - 2;
      const bool in = gi >= 0 && gi < H && gj >= 0 && gj < W;
      v[q] = in ? xb[(int64_t)gi * W + gj] : 0.f;
      if constexpr (FINE) sv[q] = in ? sb[(int64_t)gi * W + gj] : 0.f;
    }
    float ve = 0.f;
    const int re = threadIdx.x >> 2, ce = 64 + (threadIdx.x & 3), gi = i0 + re - 2, ge = j0 + ce - 2;
    if (re < LR && gi >= 0 && gi < H && ge < W) {
      ve = xb[(int64_t)gi * W + ge];
      if constexpr (FINE) ve *= sb[(int64_t)gi * W + ge];
    }
#pragma unroll
    for (int q = 0; q < LR / 4; q++) us[(wave + 4 * q) * LW + lane] = FINE ? v[q] * sv[q] : v[q];
    if (re < LR) us[re * LW + ce] = ve;
  }
  __syncthreads();
  const int ia = i0 + wave * RPT, j = j0 + lane;
  const float* ut = us + wave * RPT * LW + lane;  // row ia - 2, column j - 2
  float acc[RPT], uc[RPT];
#pragma unroll
  for (int o = 0; o < RPT; o++) acc[o] = 0.f;
#pragma unroll
  for (int r = 0; r < RPT + 4; r++) {
    float v[5];
#pragma unroll
    for (int c = 0; c < 5; c++) v[c] = ut[r * LW + c];
    if (r >= 2 && r < RPT + 2) uc[r - 2] = v[2];
#pragma unroll
    for (int o = 0; o < RPT; o++)
      if (r - o >= 0 && r - o < 5) {
#pragma unroll
        for (int c = 0; c < 5; c++) acc[o] = fmaf(st[(r - o) * 5 + c], v[c], acc[o]);
      }
  }
  if (edge) {  // the ring's own coefficients
#pragma unroll
    for (int o = 0; o < RPT; o++) {
      const int cls = edge_class(ia + o, H) * kEdge + edge_class(j, W);
      if (cls) {
        const float* sc = ring + cls * 25;
        float a = 0.f;
#pragma unroll
        for (int k = 0; k < 25; k++) a = fmaf(sc[k], ut[(o + k / 5) * LW + k % 5], a);
        acc[o] = a;
      }
    }
  }
  if (g) {  // bilinear (tent) or constant prolongation: coarse rows I, I+1 of fine row i
    const float norm = axis_norm<TENT>(f);
    const int off = TENT ? f + 1 : 0, den = TENT ? 2 * f : f;  // tent: 2i - (f-1) = 2f (I) + rem, shifted by 2f
    const int ej = TENT ? 2 * j + off : j, Jq = ej / den, J = TENT ? Jq - 1 : Jq;
    const int rj = ej - Jq * den;
    const float wj0 = TENT ? (float)(2 * f - rj) : 1.f, wj1 = (float)rj;
    const int ei = TENT ? 2 * ia + off : ia, Iq = ei / den;
    int I = TENT ? Iq - 1 : Iq, ri = ei - Iq * den;
    const float* gb = g + (int64_t)b * Hc * Wc;
    const bool in0 = J >= 0 && J < Wc, in1 = J + 1 < Wc;
    auto row = [&](int I_, float& a0, float& a1) {
      const bool rin = I_ >= 0 && I_ < Hc;
      const float* gr = gb + (int64_t)I_ * Wc + J;
      a0 = rin && in0 ? gr[0] : 0.f;
      a1 = TENT && rin && in1 && rj ? gr[1] : 0.f;
    };
    float a0, a1, b0 = 0.f, b1 = 0.f;
    row(I, a0, a1);
    if constexpr (TENT) row(I + 1, b0, b1);
#pragma unroll
    for (int o = 0; o < RPT; o++) {
      float v;
      if constexpr (TENT) {
        const float wi0 = (float)(2 * f - ri), wi1 = (float)ri;
        v = fmaf(wi0 * wj1, a1, wi0 * wj0 * a0);
        if (ri) v = fmaf(wi1 * wj1, b1, fmaf(wi1 * wj0, b0, v));
      } else {
        v = a0;
      }
      acc[o] += v * norm;
      ri += TENT ? 2 : 1;
      if (ri >= den && o + 1 < RPT) {  // the same for the whole wave
        ri -= den;
        I++;
        if constexpr (TENT) {
          a0 = b0;
          a1 = b1;
          row(I + 1, b0, b1);
        } else {
          row(I, a0, a1);
        }
      }
    }
  }
  if (j < W) {
    const float alpha = FINE ? expf(log_alpha[0]) : 0.f;
#pragma unroll
    for (int o = 0; o < RPT; o++)
      if (ia + o < H) {
        const int64_t p = (int64_t)(ia + o) * W + j;
        float v = acc[o];
        if constexpr (FINE) v = sb[p] * (alpha * uc[o] + v);
        out[(int64_t)b * H * W + p] = v;
      }
  }
}

// The coarsest levels together hold a few thousand pixels: one workgroup per
// map restricts, applies the stencils and prolongs them in LDS, in the time of
// about one launch instead of three per level (a 32^2 and an 8^2 level: 12 us
// from 49).
constexpr int kTailLevels = 8;
constexpr int kTailPix = 6144;  // all the levels of the tail; u and g of each: 48 KB

struct Tail {
  int n;  // levels
  int H[kTailLevels], W[kTailLevels], f[kTailLevels], off[kTailLevels];
};

template <bool TENT>
__global__ void __launch_bounds__(1024) level_tail_kernel(const float* __restrict__ u, const float* __restrict__ st,
                                                          Tail t, float* __restrict__ g) {
  __shared__ float us[kTailPix], gs[kTailPix], ss[kTailLevels * kStencil];
  const int tid = threadIdx.x, n0 = t.H[0] * t.W[0];
  for (int k = tid; k < t.n * kStencil; k += 1024) ss[k] = st[k];
  u += (int64_t)blockIdx.x * n0;
  g += (int64_t)blockIdx.x * n0;
  for (int k = tid; k < n0; k += 1024) us[k] = u[k];
  __syncthreads();
  for (int l = 1; l < t.n; l++) {  // a wave per coarse sample
    const int f = t.f[l], H = t.H[l - 1], W = t.W[l - 1], Hc = t.H[l], Wc = t.W[l];
    const float norm = axis_norm<TENT>(f);
    const float* xs = us + t.off[l - 1];
    for (int o = tid >> 6; o < Hc * Wc; o += 16) {
      const int I = o / Wc, J = o - I * Wc;
      const int ia = max(0, f * I - (TENT ? f / 2 : 0)), ie = min(H, f * I + (TENT ? f + f / 2 + 1 : f));
      const int ja = max(0, f * J - (TENT ? f / 2 : 0)), je = min(W, f * J + (TENT ? f + f / 2 + 1 : f));
      const int nj = je - ja, ntap = (ie - ia) * nj;
      float v = 0.f;
      for (int q = tid & 63; q < ntap; q += 64) {
        const int i = ia + q / nj, j = ja + q % nj;
        const float w = axis_w<TENT>(i, I, f) * axis_w<TENT>(j, J, f);
        if (w != 0.f) v = fmaf(w, xs[i * W + j], v);
      }
#pragma unroll
      for (int d = 32; d; d >>= 1) v += __shfl_xor(v, d);
      if ((tid & 63) == 0) us[t.off[l] + o] = v * norm;
    }
    __syncthreads();
  }
  for (int l = t.n - 1; l >= 0; l--) {
    const int H = t.H[l], W = t.W[l];
    const float* xs = us + t.off[l];
    for (int k = tid; k < H * W; k += 1024) {
      const int i = k / W, j = k - i * W;
      const float* sc = ss + l * kStencil + (edge_class(i, H) * kEdge + edge_class(j, W)) * 25;
      float a = 0.f;
#pragma unroll
      for (int q = 0; q < 25; q++) {
        const int y = i + q / 5 - 2, z = j + q % 5 - 2;
        a = fmaf(sc[q], y >= 0 && y < H && z >= 0 && z < W ? xs[y * W + z] : 0.f, a);
      }
      if (l + 1 < t.n) {
        const int f = t.f[l + 1], Hc = t.H[l + 1], Wc = t.W[l + 1];
        const float* gc = gs + t.off[l + 1];
        const int I0 = TENT ? (2 * i + f + 1) / (2 * f) - 1 : i / f, J0 = TENT ? (2 * j + f + 1) / (2 * f) - 1 : j / f;
        float v = 0.f;
        for (int I = max(I0, 0); I <= min(I0 + (TENT ? 1 : 0), Hc - 1); I++)
          for (int J = max(J0, 0); J <= min(J0 + (TENT ? 1 : 0), Wc - 1); J++) {
            const float w = axis_w<TENT>(i, I, f) * axis_w<TENT>(j, J, f);
            if (w != 0.f) v = fmaf(w, gc[I * Wc + J], v);
          }
        a += v * axis_norm<TENT>(f);
      }
      gs[t.off[l] + k] = a;
    }
    __syncthreads();
  }
  for (int k = tid; k < n0; k += 1024) g[k] = gs[k];
}

struct LevelDims {
  int H, W;
};

inline LevelDims coarser(LevelDims d, int f) { return {(int)mk::cdiv(d.H, f), (int)mk::cdiv(d.W, f)}; }

template <bool TENT>
int launch_restrict(const float* x, const float* s, LevelDims d, int f, int B, float* y, hipStream_t st) {
  const LevelDims c = coarser(d, f);
  const int nbj = (int)mk::cdiv(c.W, TENT ? 256 / f - 1 : 256 / f), per = nbj * (int)mk::cdiv(c.H, kRC);
  const unsigned grid = (unsigned)(B * per);
  if (s)
    level_restrict_kernel<TENT, true><<<grid, 256, 0, st>>>(x, s, d.H, d.W, f, c.H, c.W, nbj, per, y);
  else
    level_restrict_kernel<TENT, false><<<grid, 256, 0, st>>>(x, s, d.H, d.W, f, c.H, c.W, nbj, per, y);
  return mk::check_launch("level_restrict_kernel");
}

template <bool FINE, bool TENT, int RPT>
int launch_level_rpt(const float* x, const float* s, const float* la, const float* coef, const float* g, LevelDims d,
                     int f, int B, float* out, hipStream_t st) {
  const LevelDims c = g ? coarser(d, f) : LevelDims{1, 1};
  const int nbj = (int)mk::cdiv(d.W, 64), per = nbj * (int)mk::cdiv(d.H, 4 * RPT);
  level_kernel<FINE, TENT, RPT><<<(unsigned)(B * per), 256, 0, st>>>(x, s, la, coef, g, d.H, d.W, f, c.H, c.W, nbj,
                                                                    per, out);
  return mk::check_launch("level_kernel");
}

template <bool FINE, bool TENT>
int launch_level(const float* x, const float* s, const float* la, const float* coef, const float* g, LevelDims d,
                 int f, int B, float* out, hipStream_t st) {
  if ((int64_t)B * mk::cdiv(d.W, 64) * mk::cdiv(d.H, 32) >= 512)
    return launch_level_rpt<FINE, TENT, 8>(x, s, la, coef, g, d, f, B, out, st);
  return launch_level_rpt<FINE, TENT, 2>(x, s, la, coef, g, d, f, B, out, st);
}

template <bool TENT>
int run_levels(float* z, const float* s, const float* r, const float* la, const float* coef, int nl,
               const int32_t* steps, int B, LevelDims fine, float* work, hipStream_t st) {
  // the tail: the longest run of last levels that fits one workgroup
  int lt = nl;
  {
    int64_t pix = 0;
    for (int l = nl - 1; l >= 1; l--) {
      LevelDims d = fine;
      for (int k = 1; k <= l; k++) d = coarser(d, steps[k]);
      pix += (int64_t)d.H * d.W;
      if (pix > kTailPix || nl - l > kTailLevels) break;
      lt = l;
    }
    if (lt == nl - 1) lt = nl;  // a single level needs no tail
  }
  // u_1.. and then, on the way back, g_1.. behind them
  int rc;
  LevelDims d = fine;
  float* p = work;
  const float* src = r;
  for (int l = 1; l < nl && l <= lt; l++) {
    if ((rc = launch_restrict<TENT>(src, l == 1 ? s : nullptr, d, steps[l], B, p, st))) return rc;
    d = coarser(d, steps[l]);
    src = p;
    p += (int64_t)B * d.H * d.W;
  }
  const int last = lt < nl ? lt : nl - 1;  // the coarsest level held in memory
  const float* g = nullptr;
  if (lt < nl) {
    Tail t;
    t.n = nl - lt;
    LevelDims e = d;
    int off = 0;
    for (int k = 0; k < t.n; k++) {
      if (k) e = coarser(e, steps[lt + k]);
      t.H[k] = e.H;
      t.W[k] = e.W;
      t.f[k] = steps[lt + k];
      t.off[k] = off;
      off += e.H * e.W;
    }
    level_tail_kernel<TENT><<<(unsigned)B, 1024, 0, st>>>(src, coef + (int64_t)lt * kStencil, t, p);
    if ((rc = mk::check_launch("level_tail_kernel"))) return rc;
    g = p;
    p += (int64_t)B * d.H * d.W;
  }
  for (int l = g ? last - 1 : last; l >= 1; l--) {
    LevelDims e = fine;
    int64_t off = 0;
    for (int k = 1; k <= l; k++) {
      if (k > 1) off += (int64_t)B * e.H * e.W;
      e = coarser(e, steps[k]);
    }
    if ((rc = launch_level<false, TENT>(work + off, nullptr, nullptr, coef + (int64_t)l * kStencil, g, e,
                                        g ? steps[l + 1] : 1, B, p, st)))
      return rc;
    g = p;
    p += (int64_t)B * e.H * e.W;
  }
  return launch_level<true, TENT>(r, s, la, coef, g, fine, nl > 1 ? steps[1] : 1, B, z, st);
}

// Adam on a flat FP32 parameter vector.  Element n-1 is log(alpha); its
// gradient is alpha * dL/dalpha, taken from dalpha (FP64, on the device).
__global__ void __launch_bounds__(256) adam_kernel(float* __restrict__ p, const float* __restrict__ g,
                                                   float* __restrict__ m, float* __restrict__ v, int n,
                                                   const double* __restrict__ dalpha, float lr, float b1, float b2,
                                                   float eps, float bc1, float bc2, float gscale) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  float gk;
  if (k == n - 1)
    gk = dalpha ? (float)((double)expf(p[k]) * dalpha[0]) : 0.f;
  else
    gk = g[k];
  gk *= gscale;
  float mk_ = b1 * m[k] + (1.f - b1) * gk;
  float vk = b2 * v[k] + (1.f - b2) * gk * gk;
  m[k] = mk_;
  v[k] = vk;
  p[k] -= lr * (mk_ / bc1) / (sqrtf(vk / bc2) + eps);
}

template <int CIN, int COUT>
int launch_conv(const float* x, const float* w, float* y, const Tiling& t, int B, int accumulate, hipStream_t st) {
  int64_t grid = (int64_t)B * t.per_img;
  MK_REQUIRE(grid > 0 && grid < INT32_MAX, MK_ERR_ARG, "conv3x3: %lld tiles out of range", (long long)grid);
  conv3x3_kernel<CIN, COUT><<<(unsigned)grid, 256, 0, st>>>(x, w, y, t, accumulate);
  return mk::check_launch("conv3x3_kernel");
}

template <int CO, int CI>
int launch_wgrad(const float* a, const float* x, const Tiling& t, int B, float* part, int groups, hipStream_t st) {
  int total = B * t.per_img;
  wgrad_kernel<CO, CI><<<groups, 256, 0, st>>>(a, x, t, total, part);
  return mk::check_launch("wgrad_kernel");
}

int wgrad_groups(int B, const Tiling& t) {
  int64_t total = (int64_t)B * t.per_img;
  return (int)(total < kWgradGroups ? total : kWgradGroups);
}

bool chan_ok(int c) { return c == 1 || c == MAXC; }

}  // namespace

extern "C" int mk_conv3x3_f32(const float* x, int32_t B, int32_t Cin, int32_t H, int32_t W, const float* w,
                              int32_t Cout, int32_t dil, float* y, int32_t accumulate, void* stream) {
  MK_REQUIRE(x && w && y, MK_ERR_ARG, "conv3x3: null argument");
  MK_REQUIRE(B > 0 && H > 0 && W > 0, MK_ERR_ARG, "conv3x3: bad shape B=%d H=%d W=%d", B, H, W);
  MK_REQUIRE(chan_ok(Cin) && chan_ok(Cout), MK_ERR_ARG, "conv3x3: channels must be 1 or %d (got %d -> %d)", MAXC,
             Cin, Cout);
  MK_REQUIRE(dil >= 1 && dil <= 4096, MK_ERR_ARG, "conv3x3: dilation %d out of range", dil);
  MK_REQUIRE((int64_t)B * Cin * H * W < ((int64_t)1 << 40), MK_ERR_ARG, "conv3x3: tensor too large");
  MK_REQUIRE(x != y, MK_ERR_ARG, "conv3x3 cannot run in place");
  Tiling t = make_tiling(H, W, dil);
  hipStream_t st = mk::as_stream(stream);
  if (Cin == 1 && Cout == MAXC) return launch_conv<1, MAXC>(x, w, y, t, B, accumulate, st);
  if (Cin == MAXC && Cout == MAXC) return launch_conv<MAXC, MAXC>(x, w, y, t, B, accumulate, st);
  if (Cin == MAXC && Cout == 1) return launch_conv<MAXC, 1>(x, w, y, t, B, accumulate, st);
  return launch_conv<1, 1>(x, w, y, t, B, accumulate, st);
}

extern "C" int mk_conv3x3_adjoint_weights(const float* w, int32_t Co, int32_t Ci, float* wt, void* stream) {
  MK_REQUIRE(w && wt && w != wt, MK_ERR_ARG, "adjoint_weights: bad pointers");
  MK_REQUIRE(Co >= 1 && Co <= MAXC && Ci >= 1 && Ci <= MAXC, MK_ERR_ARG, "adjoint_weights: bad channels");
  int nw = Co * Ci * 9;
  adjoint_weights_kernel<<<(unsigned)mk::cdiv(nw, 256), 256, 0, mk::as_stream(stream)>>>(w, Co, Ci, wt);
  return mk::check_launch("adjoint_weights_kernel");
}

extern "C" int64_t mk_conv3x3_wgrad_workspace_bytes(int32_t B, int32_t Co, int32_t Ci, int32_t H, int32_t W,
                                                    int32_t dil) {
  if (B <= 0 || H <= 0 || W <= 0 || dil < 1 || Co < 1 || Ci < 1) return -1;
  Tiling t = make_tiling(H, W, dil);
  return (int64_t)wgrad_groups(B, t) * Co * Ci * 9 * 4 + 256;
}

extern "C" int mk_conv3x3_wgrad_f32(const float* a, int32_t Co, const float* x, int32_t Ci, int32_t B, int32_t H,
                                    int32_t W, int32_t dil, float* g, int32_t accumulate, void* work,
                                    int64_t work_bytes, void* stream) {
  MK_REQUIRE(a && x && g && work, MK_ERR_ARG, "wgrad: null argument");
  MK_REQUIRE(chan_ok(Co) && chan_ok(Ci) && B > 0 && H > 0 && W > 0, MK_ERR_ARG, "wgrad: bad shape");
  MK_REQUIRE(dil >= 1 && dil <= 4096, MK_ERR_ARG, "wgrad: dilation %d out of range", dil);
  MK_REQUIRE((int64_t)B * MAXC * H * W < ((int64_t)1 << 40), MK_ERR_ARG, "wgrad: tensor too large");
  MK_REQUIRE(work_bytes >= mk_conv3x3_wgrad_workspace_bytes(B, Co, Ci, H, W, dil), MK_ERR_ARG,
             "wgrad: workspace too small");
  Tiling t = make_tiling(H, W, dil);
  MK_REQUIRE((int64_t)B * t.per_img < INT32_MAX, MK_ERR_ARG, "wgrad: too many tiles");
  int groups = wgrad_groups(B, t);
  hipStream_t st = mk::as_stream(stream);
  float* part = (float*)work;
  int r;
  if (Co == MAXC && Ci == MAXC) r = launch_wgrad<MAXC, MAXC>(a, x, t, B, part, groups, st);
  else if (Co == MAXC && Ci == 1) r = launch_wgrad<MAXC, 1>(a, x, t, B, part, groups, st);
  else if (Co == 1 && Ci == MAXC) r = launch_wgrad<1, MAXC>(a, x, t, B, part, groups, st);
  else r = launch_wgrad<1, 1>(a, x, t, B, part, groups, st);
  if (r) return r;
  int nw = Co * Ci * 9;
  wgrad_reduce_kernel<<<(unsigned)mk::cdiv(nw, 256), 256, 0, st>>>(part, groups, nw, g, accumulate);
  return mk::check_launch("wgrad_reduce_kernel");
}

extern "C" int mk_precon_finish_f32(float* z, const float* s, const float* log_alpha, const float* u, const float* g,
                                    int64_t n, void* stream) {
  MK_REQUIRE(z && s && log_alpha && u && n >= 0, MK_ERR_ARG, "precon_finish: null argument");
  if (n == 0) return MK_OK;
  precon_finish_kernel<<<mk::grid_for(n, 256), 256, 0, mk::as_stream(stream)>>>(z, s, log_alpha, u, g, n);
  return mk::check_launch("precon_finish_kernel");
}

extern "C" int64_t mk_precon_loss_workspace_bytes(void) { return (int64_t)2 * kLossGroups * sizeof(double); }

extern "C" int mk_precon_loss_f32(const float* g, const float* u, const float* s, const float* e, const float* m,
                                  const float* log_alpha, int64_t n, float* q, double* sc, void* work,
                                  int64_t work_bytes, void* stream) {
  MK_REQUIRE(g && u && s && e && m && log_alpha && q && sc && work, MK_ERR_ARG, "precon_loss: null argument");
  MK_REQUIRE(n > 0, MK_ERR_ARG, "precon_loss: empty input");
  MK_REQUIRE(work_bytes >= mk_precon_loss_workspace_bytes(), MK_ERR_ARG, "precon_loss: workspace too small");
  hipStream_t st = mk::as_stream(stream);
  precon_loss_stage1<<<kLossGroups, 256, 0, st>>>(g, u, s, e, m, log_alpha, n, q, (double*)work);
  int r = mk::check_launch("precon_loss_stage1");
  if (r) return r;
  precon_loss_stage2<<<1, 256, 0, st>>>((const double*)work, sc);
  return mk::check_launch("precon_loss_stage2");
}

extern "C" int mk_adam_f32(float* p, const float* g, float* m, float* v, int32_t n, const double* dalpha, float lr,
                           float beta1, float beta2, float eps, int32_t step, float gscale, void* stream) {
  MK_REQUIRE(p && g && m && v && n > 0 && step >= 1, MK_ERR_ARG, "adam: bad argument");
  float bc1 = 1.f - powf(beta1, (float)step), bc2 = 1.f - powf(beta2, (float)step);
  adam_kernel<<<(unsigned)mk::cdiv(n, 256), 256, 0, mk::as_stream(stream)>>>(p, g, m, v, n, dalpha, lr, beta1, beta2,
                                                                            eps, bc1, bc2, gscale);
  return mk::check_launch("adam_kernel");
}

extern "C" int mk_precon_aloss_f32(const float* z, const float* az, const float* r, const float* e, const float* s,
                                   const float* u, int64_t n, float* q, double* sc, void* work, int64_t work_bytes,
                                   void* stream) {
  MK_REQUIRE(z && az && r && e && s && u && q && sc && work, MK_ERR_ARG, "precon_aloss: null argument");
  MK_REQUIRE(n > 0, MK_ERR_ARG, "precon_aloss: empty input");
  MK_REQUIRE(work_bytes >= mk_precon_loss_workspace_bytes(), MK_ERR_ARG, "precon_aloss: workspace too small");
  hipStream_t st = mk::as_stream(stream);
  precon_aloss_stage1<<<kLossGroups, 256, 0, st>>>(z, az, r, e, s, u, n, q, (double*)work);
  int rc = mk::check_launch("precon_aloss_stage1");
  if (rc) return rc;
  precon_loss_stage2<<<1, 256, 0, st>>>((const double*)work, sc);
  return mk::check_launch("precon_loss_stage2");
}

extern "C" int mk_restrict_box_f32(const float* x, int32_t B, int32_t H, int32_t W, int32_t f, float* y, void* stream) {
  MK_REQUIRE(x && y && x != y, MK_ERR_ARG, "restrict: bad pointers");
  MK_REQUIRE(B > 0 && H > 0 && W > 0 && f >= 1 && f <= 64, MK_ERR_ARG, "restrict: bad shape");
  int Hc = (int)mk::cdiv(H, f), Wc = (int)mk::cdiv(W, f);
  int64_t total = (int64_t)B * Hc * Wc;
  restrict_kernel<<<mk::grid_for(total, 256), 256, 0, mk::as_stream(stream)>>>(x, H, W, f, Hc, Wc, total, y);
  return mk::check_launch("restrict_kernel");
}

extern "C" int mk_prolong_box_f32(const float* y, int32_t B, int32_t H, int32_t W, int32_t f, float* x,
                                  int32_t accumulate, void* stream) {
  MK_REQUIRE(x && y && x != y, MK_ERR_ARG, "prolong: bad pointers");
  MK_REQUIRE(B > 0 && H > 0 && W > 0 && f >= 1 && f <= 64, MK_ERR_ARG, "prolong: bad shape");
  int Hc = (int)mk::cdiv(H, f), Wc = (int)mk::cdiv(W, f);
  int64_t total = (int64_t)B * H * W;
  prolong_kernel<<<mk::grid_for(total, 256), 256, 0, mk::as_stream(stream)>>>(y, Hc, Wc, f, H, W, total, x,
                                                                               accumulate);
  return mk::check_launch("prolong_kernel");
}

extern "C" int mk_restrict_tent_f32(const float* x, int32_t B, int32_t H, int32_t W, int32_t f, float* y,
                                    void* stream) {
  MK_REQUIRE(x && y && x != y, MK_ERR_ARG, "restrict_tent: bad pointers");
  MK_REQUIRE(B > 0 && H > 0 && W > 0 && f >= 1 && f <= 64, MK_ERR_ARG, "restrict_tent: bad shape");
  int Hc = (int)mk::cdiv(H, f), Wc = (int)mk::cdiv(W, f);
  int64_t total = (int64_t)B * Hc * Wc;
  restrict_tent_kernel<<<mk::grid_for(total, 256), 256, 0, mk::as_stream(stream)>>>(x, H, W, f, Hc, Wc, total, y);
  return mk::check_launch("restrict_tent_kernel");
}

extern "C" int mk_prolong_tent_f32(const float* y, int32_t B, int32_t H, int32_t W, int32_t f, float* x,
                                   int32_t accumulate, void* stream) {
  MK_REQUIRE(x && y && x != y, MK_ERR_ARG, "prolong_tent: bad pointers");
  MK_REQUIRE(B > 0 && H > 0 && W > 0 && f >= 1 && f <= 64, MK_ERR_ARG, "prolong_tent: bad shape");
  int Hc = (int)mk::cdiv(H, f), Wc = (int)mk::cdiv(W, f);
  int64_t total = (int64_t)B * H * W;
  prolong_tent_kernel<<<mk::grid_for(total, 256), 256, 0, mk::as_stream(stream)>>>(y, Hc, Wc, f, H, W, total, x,
                                                                                    accumulate);
  return mk::check_launch("prolong_tent_kernel");
}

extern "C" int64_t mk_level_stencils_floats(int32_t nlevel) { return nlevel < 1 ? -1 : (int64_t)nlevel * kStencil; }

extern "C" int mk_level_stencils_f32(const float* w, int32_t nlevel, float* st, void* stream) {
  MK_REQUIRE(w && st && nlevel >= 1 && nlevel <= 65535, MK_ERR_ARG, "level_stencils: bad argument");
  level_stencil_kernel<<<(unsigned)nlevel, 256, 0, mk::as_stream(stream)>>>(w, st);
  return mk::check_launch("level_stencil_kernel");
}

namespace {
bool levels_ok(int32_t nlevel, const int32_t* steps, int32_t B, int32_t H, int32_t W) {
  if (nlevel < 1 || !steps || B < 1 || H < 1 || W < 1) return false;
  for (int l = 1; l < nlevel; l++)
    if (steps[l] < 1 || steps[l] > 64) return false;
  // the finest tiling is the largest grid: restriction by up to 64 (3 coarse
  // columns of a workgroup) and 64 x 8 pixel tiles
  return (int64_t)B * (mk::cdiv(W, 64) + 1) * (mk::cdiv(H, 4) + 1) < INT32_MAX;
}
}  // namespace

extern "C" int64_t mk_precon_levels_workspace_bytes(int32_t nlevel, const int32_t* steps, int32_t B, int32_t H,
                                                    int32_t W) {
  if (!levels_ok(nlevel, steps, B, H, W)) return -1;
  int64_t n = 0;
  LevelDims d{H, W};
  for (int l = 1; l < nlevel; l++) {
    d = coarser(d, steps[l]);
    n += (int64_t)2 * B * d.H * d.W;
  }
  return n * 4;
}

extern "C" int mk_precon_levels_f32(float* z, const float* s, const float* r, const float* log_alpha,
                                    const float* stencils, int32_t tent, int32_t nlevel, const int32_t* steps,
                                    int32_t B, int32_t H, int32_t W, void* work, int64_t work_bytes, void* stream) {
  MK_REQUIRE(z && s && r && log_alpha && stencils, MK_ERR_ARG, "precon_levels: null argument");
  MK_REQUIRE(levels_ok(nlevel, steps, B, H, W), MK_ERR_ARG, "precon_levels: bad shape");
  const int64_t n = (int64_t)B * H * W, need = mk_precon_levels_workspace_bytes(nlevel, steps, B, H, W);
  MK_REQUIRE(need == 0 || (work && work_bytes >= need), MK_ERR_ARG, "precon_levels: workspace too small");
  MK_REQUIRE((z + n <= r || r + n <= z) && (z + n <= s || s + n <= z), MK_ERR_ARG,
             "precon_levels: z overlaps an input");
  hipStream_t st = mk::as_stream(stream);
  const LevelDims d{H, W};
  return tent ? run_levels<true>(z, s, r, log_alpha, stencils, nlevel, steps, B, d, (float*)work, st)
              : run_levels<false>(z, s, r, log_alpha, stencils, nlevel, steps, B, d, (float*)work, st);
}
