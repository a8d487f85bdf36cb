// TOD preprocessing of minkasi's canonical pipeline
// (examples/minkasi_mpi_example.py:42-52): fit_cm_plus_poly
// (minkasi/tods/processing.py:510-579), the common-mode median over
// detectors plus a least-squares fit of Legendre drifts and the Legendre-
// weighted common mode (_linfit_2mat, processing.py:28-39).
//
//  median_cols   : per sample (column) the median over the detectors (rows),
//                  numpy semantics (mean of the two middle values for an even
//                  count, NaN if the column holds one), as exact order
//                  statistics of the values' ordered bit patterns: one wave
//                  per column bisects on them, or sorts up to 64.
//  design        : X[t][k] = P_k(x_t) (k <= ord) and X[t][ord+1+i] =
//                  P_i(x_t) cm[t] (i < cm_ord), x_t = (t - (n-1)/2) / ((n-1)/2),
//                  Legendre P by the three-term recurrence, FP64; also X^T.
//  design_dots   : D[k][j] = sum_t X[t][k] y_j[t] for rows y_j, FP64, per-row
//                  chunk partials summed in a fixed order.
//  design_apply  : out[j][t] = base[j][t] - sum_k X[t][c0+k] coef[k][j] (or
//                  the plain product without base).
#include "common.h"

#include <algorithm>
#include <cmath>

namespace {

constexpr int kWave = 64;

// Bit patterns whose unsigned order is the order of the values.
__device__ __forceinline__ uint32_t order_key(float v) {
  const uint32_t u = __float_as_uint(v);
  return u ^ ((u >> 31) ? 0xffffffffu : 0x80000000u);
}
__device__ __forceinline__ uint64_t order_key(double v) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  return u ^ ((u >> 63) ? ~0ull : 1ull << 63);
}
__device__ __forceinline__ float key_value(uint32_t k) {
  return __uint_as_float(k ^ ((k >> 31) ? 0x80000000u : 0xffffffffu));
}
__device__ __forceinline__ double key_value(uint64_t k) {
  return __longlong_as_double((long long)(k ^ ((k >> 63) ? 1ull << 63 : ~0ull)));
}
template <typename T>
struct KeyOf;
template <>
struct KeyOf<float> { using type = uint32_t; };
template <>
struct KeyOf<double> { using type = uint64_t; };

// Whether a column whose smallest and largest keys are these holds a NaN: its
// key lies above +inf's or below -inf's.
template <typename T>
__device__ __forceinline__ bool has_nan(typename KeyOf<T>::type lo, typename KeyOf<T>::type hi) {
  return hi > order_key((T)INFINITY) || lo < order_key((T)-INFINITY);
}

// Smallest of the wave, in scalar registers.
__device__ __forceinline__ uint32_t wave_min(uint32_t v) {
#pragma unroll
  for (int d = 32; d; d >>= 1) v = min(v, (uint32_t)__shfl_xor((int)v, d, 64));
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}
__device__ __forceinline__ uint64_t wave_min(uint64_t v) {
#pragma unroll
  for (int d = 32; d; d >>= 1) v = min(v, (uint64_t)__shfl_xor((unsigned long long)v, d, 64));
  return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v) |
         (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32;
}

// v of lane l ^ d.  Moves by 1, 2 and 8 stay within a row of 16 lanes and the
// vector unit makes them; ds_bpermute, which the others take, is what a sort
// would be bound by.
__device__ __forceinline__ uint32_t lane_xor(uint32_t v, int d) {
  if (d == 1) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, true);   // quad 1 0 3 2
  if (d == 2) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4e, 0xf, 0xf, true);   // quad 2 3 0 1
  if (d == 8) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xf, 0xf, true);  // row rotated by 8
  return (uint32_t)__shfl_xor((int)v, d, 64);
}
__device__ __forceinline__ uint64_t lane_xor(uint64_t v, int d) {
  return (uint64_t)lane_xor((uint32_t)v, d) | (uint64_t)lane_xor((uint32_t)(v >> 32), d) << 32;
}
// Lane l's value (l uniform), in scalar registers.
__device__ __forceinline__ uint32_t lane_value(uint32_t v, int l) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}
__device__ __forceinline__ uint64_t lane_value(uint64_t v, int l) {
  return (uint64_t)lane_value((uint32_t)v, l) | (uint64_t)lane_value((uint32_t)(v >> 32), l) << 32;
}

// Bitonic sort of one key per lane, ascending.
template <typename K>
__device__ __forceinline__ K wave_sort(K x, int lane) {
#pragma unroll
  for (int k = 2; k <= kWave; k <<= 1) {
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1) {
      const K y = lane_xor(x, j);
      const bool low = ((lane & k) == 0) == ((lane & j) == 0);  // this lane takes the smaller one
      x = (x < y) == low ? x : y;
    }
  }
  return x;
}

// Bound by the scalar work of the bisection.  A workgroup stages C columns
// through LDS, so rows are read along their length (a wave per column would
// fetch a line for every value), and a wave then holds a column in V registers
// a lane.  A step counts the keys up to a pivot with one compare and one
// population count of the lane mask per register; the bracket starts at the
// smallest and largest key and closes as soon as one key is left in it, so a
// column takes about log2(nrow) steps more than its values share leading bits,
// against (6 + log2 V)(7 + log2 V)/2 exchange stages of a full sort.  215 x
// 100003 FP32: 65 us from 151 us (bitonic sort over lanes and registers, column
// loads).  Up to 64 rows the 21 stages of a sort, one key a lane, cost less than
// the bisection's dependent steps: 64 x 100003 21 us FP32 and 31 us FP64, the
// bisection 42 and 59.
template <typename T, int V>
__global__ void __launch_bounds__(256) median_cols_kernel(const T* __restrict__ dat, int64_t nrow, int64_t ncol,
                                                          int64_t ld, int cbits, T* __restrict__ out) {
  using K = typename KeyOf<T>::type;
  extern __shared__ __align__(8) unsigned char lds[];
  K* tile = (K*)lds;  // [column][row], odd pitch
  const int n = (int)nrow, pitch = n | 1, C = 1 << cbits;
  const int64_t c0 = (int64_t)blockIdx.x << cbits;
  const int cq = threadIdx.x & (C - 1), rstep = 256 >> cbits;
  if (c0 + cq < ncol) {
    const T* p = dat + c0 + cq;
#pragma unroll 8
    for (int i = threadIdx.x >> cbits; i < n; i += rstep) tile[cq * pitch + i] = order_key(p[(int64_t)i * ld]);
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int ncl = (int)min((int64_t)C, ncol - c0);
  const int k = (n - 1) / 2;  // the lower middle value
  for (int c = threadIdx.x >> 6; c < ncl; c += 4) {
    if constexpr (V == 1) {
      const K x = wave_sort(lane < n ? tile[c * pitch + lane] : ~(K)0, lane);  // the padding sorts last
      const K first = lane_value(x, 0), last = lane_value(x, n - 1);
      T med = key_value(lane_value(x, k));
      if (!(n & 1)) med = (med + key_value(lane_value(x, n / 2))) / T(2);
      if (lane == 0) out[c0 + c] = has_nan<T>(first, last) ? (T)NAN : med;
      continue;
    }
    K x[V];
    K mn = ~(K)0, mx = 0;
#pragma unroll
    for (int e = 0; e < V; e++) {
      const int i = e * kWave + lane;
      const bool in = i < n;
      x[e] = in ? tile[c * pitch + i] : ~(K)0;  // the padding counts only above every pivot
      mn = min(mn, x[e]);
      mx = max(mx, in ? x[e] : (K)0);
    }
    K lo = wave_min(mn), hi = ~wave_min((K)~mx);  // x_k is in [lo, hi]
    const bool nan = has_nan<T>(lo, hi);
    int clo = 0, chi = n;                         // keys below lo, keys up to hi
    while (lo < hi && chi - clo > 1) {
      const K mid = lo + (hi - lo) / 2;
      int cnt = 0;
#pragma unroll
      for (int e = 0; e < V; e++) cnt += __popcll(__ballot(x[e] <= mid));
      if (cnt > k) {
        hi = mid;
        chi = cnt;
      } else {
        lo = mid + 1;
        clo = cnt;
      }
    }
    K a = hi;
    if (lo < hi) {  // the one key in the bracket
      a = ~(K)0;
#pragma unroll
      for (int e = 0; e < V; e++) a = min(a, x[e] >= lo ? x[e] : ~(K)0);
      a = wave_min(a);
    }
    T med = key_value(a);
    if (!(n & 1)) {
      K b = a;
      if (chi < k + 2) {  // the next value up is another one
        b = ~(K)0;
#pragma unroll
        for (int e = 0; e < V; e++) b = min(b, x[e] > a ? x[e] : ~(K)0);
        b = wave_min(b);
      }
      med = (med + key_value(b)) / T(2);
    }
    if (lane == 0) out[c0 + c] = nan ? (T)NAN : med;
  }
}

template <typename T>
__global__ void __launch_bounds__(256) design_kernel(const T* __restrict__ cm, int64_t n, int ord, int cm_ord,
                                                     double* __restrict__ X, double* __restrict__ Xt) {
  const int ncol = ord + 1 + cm_ord;
  const double half = 0.5 * (double)(n - 1);
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x) {
    const double x = ((double)t - half) / half;
    const int kmax = ord > cm_ord - 1 ? ord : cm_ord - 1;
    double pm2 = 1.0, pm1 = x;
    const double c = (double)cm[t];
    for (int k = 0; k <= kmax; k++) {
      double p;
      if (k == 0) p = 1.0;
      else if (k == 1) p = x;
      else {
        p = (pm1 * x * (2 * k - 1) - pm2 * (k - 1)) / k;
        pm2 = pm1;
        pm1 = p;
      }
      if (k <= ord) {
        X[t * ncol + k] = p;
        Xt[k * n + t] = p;
      }
      if (k < cm_ord) {
        X[t * ncol + ord + 1 + k] = p * c;
        Xt[(int64_t)(ord + 1 + k) * n + t] = p * c;
      }
    }
  }
}

constexpr int kMaxCol = 8;
constexpr int kDotRows = 8;  // rows per workgroup

// Samples per partial: 4096, down to 512 while two workgroups a CU are not
// filled.  64 x 50000 FP32: 38 us at 4096, 17 at 512; 215 x 100003: 50 at
// 4096, 71 at 512.
constexpr int64_t kDotChunk = 4096, kDotChunkMin = 512, kDotGroups = 512;

int64_t dot_chunk(int64_t n, int64_t nrow) {
  int64_t chunk = kDotChunk;
  while (chunk > kDotChunkMin && mk::cdiv(nrow, kDotRows) * mk::cdiv(n, chunk) < kDotGroups) chunk /= 2;
  return chunk;
}

// part[(j * nchunk + chunk) * ncol + k] = sum over the chunk of X[t][k] y_j[t].
// Bandwidth-bound on y: a thread holds one sample's NC design values and
// applies them to kDotRows rows, so the FP64 design, twice as wide as a FP32
// row per column, is read once per 8 rows instead of once per row.  The 8 x NC
// sums of a thread are halved and exchanged lane by lane, after which lane l
// holds sum l of the wave (63 exchanges instead of 6 per sum).  215 rows x
// 100003, NC = 6, FP32: 47 us from 247 us (a row per workgroup).
template <typename T, int NC>
__global__ void __launch_bounds__(256) design_dots_kernel(const double* __restrict__ X, int64_t n,
                                                          const T* __restrict__ y, int64_t nrow, int64_t ld,
                                                          int64_t nchunk, int64_t len, double* __restrict__ part) {
  __shared__ double red[4][64];
  const int64_t j0 = (int64_t)blockIdx.y * kDotRows, chunk = blockIdx.x;
  const int64_t t0 = chunk * len, t1 = min(n, t0 + len);
  const int nr = (int)min((int64_t)kDotRows, nrow - j0);
  double acc[64];
#pragma unroll
  for (int e = 0; e < 64; e++) acc[e] = 0.0;
  const T* rows = y + j0 * ld;
#pragma unroll 2
  for (int64_t t = t0 + threadIdx.x; t < t1; t += 256) {
    double xv[NC];
    T v[kDotRows];
#pragma unroll
    for (int r = 0; r < kDotRows; r++) v[r] = r < nr ? rows[r * ld + t] : T(0);
#pragma unroll
    for (int k = 0; k < NC; k++) xv[k] = X[t * NC + k];
#pragma unroll
    for (int r = 0; r < kDotRows; r++)
#pragma unroll
      for (int k = 0; k < NC; k++) acc[r * 8 + k] += xv[k] * (double)v[r];
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int h = 32; h; h >>= 1) {
    const bool up = lane & h;
#pragma unroll
    for (int e = 0; e < h; e++) {
      const double keep = up ? acc[e + h] : acc[e], give = up ? acc[e] : acc[e + h];
      acc[e] = keep + __shfl_xor(give, h, 64);
    }
  }
  red[wave][lane] = acc[0];
  __syncthreads();
  const int r = threadIdx.x >> 3, k = threadIdx.x & 7;
  if (r < nr && k < NC)
    part[((j0 + r) * nchunk + chunk) * NC + k] = ((red[0][threadIdx.x] + red[1][threadIdx.x]) + red[2][threadIdx.x]) +
                                                 red[3][threadIdx.x];
}

// D[k][j] = sum over chunks of the partials, a wave per sum: lane l adds chunks
// l, l + 64, ... and the lanes' sums are added in a fixed order, so that the
// many short chunks of a small block do not queue behind one thread's loads.
__global__ void __launch_bounds__(256) design_dots_reduce(const double* __restrict__ part, int64_t nrow, int ncol,
                                                          int64_t nchunk, double* __restrict__ D) {
  const int64_t e = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (e >= nrow * ncol) return;  // whole wave
  const int64_t j = e / ncol, k = e % ncol;
  double s = 0.0;
  for (int64_t c = threadIdx.x & 63; c < nchunk; c += 64) s += part[(j * nchunk + c) * ncol + k];
#pragma unroll
  for (int d = 32; d; d >>= 1) s += __shfl_xor(s, d, 64);
  if ((threadIdx.x & 63) == 0) D[k * nrow + j] = s;
}

// Bandwidth-bound on base and out: a thread holds one sample's NK design
// values and applies them to kDotRows rows, whose coefficients are scalar.
// 215 x 100003, NK = 3, FP32: 50 us (3.4 TB/s) from 120 us (one element per thread and
// step, the design read again for every row).  NK < 0: more than kMaxCol
// columns, read as they are used.
template <typename T, int NK>
__global__ void __launch_bounds__(256) design_apply_kernel(const T* __restrict__ base, int64_t nrow, int64_t n,
                                                           int64_t ld, const double* __restrict__ X, int ncol, int c0,
                                                           int nk, const double* __restrict__ coef,
                                                           T* __restrict__ out, int64_t ld_out, int64_t ntile) {
  const int64_t jg = blockIdx.x / ntile, t = (blockIdx.x - jg * ntile) * 256 + threadIdx.x;
  if (t >= n) return;
  const int64_t j0 = jg * kDotRows;
  const int nr = (int)min((int64_t)kDotRows, nrow - j0);
  double xv[NK > 0 ? NK : 1];
#pragma unroll
  for (int k = 0; k < NK; k++) xv[k] = X[t * ncol + c0 + k];
  T v[kDotRows];
#pragma unroll
  for (int r = 0; r < kDotRows; r++) v[r] = base && r < nr ? base[(j0 + r) * ld + t] : T(0);
#pragma unroll
  for (int r = 0; r < kDotRows; r++) {
    if (r >= nr) break;
    double p = 0.0;
#pragma unroll
    for (int k = 0; k < NK; k++) p += xv[k] * coef[k * nrow + j0 + r];
    if constexpr (NK < 0)
      for (int k = 0; k < nk; k++) p += X[t * ncol + c0 + k] * coef[k * nrow + j0 + r];
    out[(j0 + r) * ld_out + t] = base ? (T)((double)v[r] - p) : (T)p;
  }
}

template <typename T>
int median_cols_impl(const T* dat, int64_t nrow, int64_t ncol, int64_t ld, T* out, void* stream) {
  MK_REQUIRE(nrow >= 1 && nrow <= 1024 && ncol >= 0 && ld >= ncol, MK_ERR_ARG,
             "median over 1..1024 rows (got %lld rows, %lld columns, ld %lld)", (long long)nrow, (long long)ncol,
             (long long)ld);
  if (ncol == 0) return MK_OK;
  MK_REQUIRE(dat && out, MK_ERR_ARG, "null pointer");
  // Columns per workgroup: up to 32, while they fit 20 KB (eight workgroups a
  // CU) and leave four workgroups a CU; at least one for each wave.
  // 64 x 4000 FP32 takes 5.8 us with 4 columns a workgroup, 14 with 32; 64 x
  // 100003 37 us with 4, 30 with 32 (sorted without row moves).
  int cbits = 5;
  while (cbits > 2 && ((((size_t)(nrow | 1) * sizeof(T)) << cbits) > 20 * 1024 || (ncol >> cbits) < 1024)) cbits--;
  const size_t lds = ((size_t)(nrow | 1) * sizeof(T)) << cbits;
  const int64_t groups = mk::cdiv(ncol, (int64_t)1 << cbits);
  MK_REQUIRE(groups < INT32_MAX, MK_ERR_ARG, "median: too many columns");
  const unsigned grid = (unsigned)groups;
  hipStream_t st = mk::as_stream(stream);
  if (nrow <= 64) median_cols_kernel<T, 1><<<grid, 256, lds, st>>>(dat, nrow, ncol, ld, cbits, out);
  else if (nrow <= 128) median_cols_kernel<T, 2><<<grid, 256, lds, st>>>(dat, nrow, ncol, ld, cbits, out);
  else if (nrow <= 256) median_cols_kernel<T, 4><<<grid, 256, lds, st>>>(dat, nrow, ncol, ld, cbits, out);
  else if (nrow <= 512) median_cols_kernel<T, 8><<<grid, 256, lds, st>>>(dat, nrow, ncol, ld, cbits, out);
  else median_cols_kernel<T, 16><<<grid, 256, lds, st>>>(dat, nrow, ncol, ld, cbits, out);
  return mk::check_launch("median_cols_kernel");
}

template <typename T>
int design_impl(const T* cm, int64_t n, int ord, int cm_ord, double* X, double* Xt, void* stream) {
  MK_REQUIRE(n >= 2 && ord >= 0 && cm_ord >= 0 && ord + 1 + cm_ord <= kMaxCol, MK_ERR_ARG,
             "design needs n >= 2 and ord + 1 + cm_ord <= %d", kMaxCol);
  MK_REQUIRE(cm && X && Xt, MK_ERR_ARG, "null pointer");
  design_kernel<T><<<mk::grid_for(n, 256), 256, 0, mk::as_stream(stream)>>>(cm, n, ord, cm_ord, X, Xt);
  return mk::check_launch("design_kernel");
}

template <typename T>
int dots_impl(const double* X, int64_t n, int ncol, const T* y, int64_t nrow, int64_t ld, double* D, void* work,
              int64_t work_bytes, void* stream) {
  MK_REQUIRE(n >= 1 && ncol >= 1 && ncol <= kMaxCol && nrow >= 1 && nrow < 65536 && ld >= n, MK_ERR_ARG,
             "bad design dot sizes");
  MK_REQUIRE(X && y && D && work, MK_ERR_ARG, "null pointer");
  const int64_t chunk = dot_chunk(n, nrow), nchunk = mk::cdiv(n, chunk);
  MK_REQUIRE(work_bytes >= nrow * nchunk * ncol * 8, MK_ERR_ARG, "workspace too small");
  hipStream_t st = mk::as_stream(stream);
  const dim3 grid((unsigned)nchunk, (unsigned)mk::cdiv(nrow, kDotRows));
  double* part = (double*)work;
  switch (ncol) {
#define MK_DOTS(NC) \
  case NC: design_dots_kernel<T, NC><<<grid, 256, 0, st>>>(X, n, y, nrow, ld, nchunk, chunk, part); break
    MK_DOTS(1); MK_DOTS(2); MK_DOTS(3); MK_DOTS(4); MK_DOTS(5); MK_DOTS(6); MK_DOTS(7); MK_DOTS(8);
#undef MK_DOTS
  }
  int r = mk::check_launch("design_dots_kernel");
  if (r) return r;
  design_dots_reduce<<<(unsigned)mk::cdiv(nrow * ncol, 4), 256, 0, st>>>((const double*)work, nrow, ncol, nchunk, D);
  return mk::check_launch("design_dots_reduce");
}

template <typename T>
int apply_impl(const T* base, int64_t nrow, int64_t n, int64_t ld, const double* X, int ncol, int c0, int nk,
               const double* coef, T* out, int64_t ld_out, void* stream) {
  MK_REQUIRE(nrow >= 0 && n >= 1 && ncol >= 1 && c0 >= 0 && nk >= 0 && c0 + nk <= ncol && ld >= n && ld_out >= n,
             MK_ERR_ARG, "bad design apply sizes");
  if (nrow == 0) return MK_OK;
  MK_REQUIRE(X && coef && out, MK_ERR_ARG, "null pointer");
  const int64_t ntile = mk::cdiv(n, 256), groups = ntile * mk::cdiv(nrow, kDotRows);
  MK_REQUIRE(groups < INT32_MAX, MK_ERR_ARG, "bad design apply sizes");
  hipStream_t st = mk::as_stream(stream);
  switch (nk) {
#define MK_APPLY(LABEL, NK)                                                                                      \
  LABEL:                                                                                                         \
    design_apply_kernel<T, NK><<<(unsigned)groups, 256, 0, st>>>(base, nrow, n, ld, X, ncol, c0, nk, coef, out,  \
                                                                 ld_out, ntile);                                 \
    break
    MK_APPLY(case 0, 0); MK_APPLY(case 1, 1); MK_APPLY(case 2, 2); MK_APPLY(case 3, 3); MK_APPLY(case 4, 4);
    MK_APPLY(case 5, 5); MK_APPLY(case 6, 6); MK_APPLY(case 7, 7); MK_APPLY(case 8, 8); MK_APPLY(default, -1);
#undef MK_APPLY
  }
  return mk::check_launch("design_apply_kernel");
}

}  // namespace

extern "C" int mk_median_cols_f32(const float* dat, int64_t nrow, int64_t ncol, int64_t ld, float* out,
                                  void* stream) {
  return median_cols_impl<float>(dat, nrow, ncol, ld, out, stream);
}
extern "C" int mk_median_cols_f64(const double* dat, int64_t nrow, int64_t ncol, int64_t ld, double* out,
                                  void* stream) {
  return median_cols_impl<double>(dat, nrow, ncol, ld, out, stream);
}
extern "C" int mk_cm_poly_design_f32(const float* cm, int64_t n, int ord, int cm_ord, double* X, double* Xt,
                                     void* stream) {
  return design_impl<float>(cm, n, ord, cm_ord, X, Xt, stream);
}
extern "C" int mk_cm_poly_design_f64(const double* cm, int64_t n, int ord, int cm_ord, double* X, double* Xt,
                                     void* stream) {
  return design_impl<double>(cm, n, ord, cm_ord, X, Xt, stream);
}
extern "C" int64_t mk_design_dots_workspace_bytes(int64_t n, int ncol, int64_t nrow) {
  // Never less for a smaller n or nrow, so that the size for the largest call
  // serves the others: 8 rows of at most 2 kDotGroups shorter chunks.
  return std::max(nrow * mk::cdiv(n, kDotChunk),
                  std::min(nrow * mk::cdiv(n, kDotChunkMin), 2 * kDotGroups * kDotRows)) *
             ncol * 8 +
         256;
}
extern "C" int mk_design_dots_f32(const double* X, int64_t n, int ncol, const float* y, int64_t nrow, int64_t ld,
                                  double* D, void* work, int64_t work_bytes, void* stream) {
  return dots_impl<float>(X, n, ncol, y, nrow, ld, D, work, work_bytes, stream);
}
extern "C" int mk_design_dots_f64(const double* X, int64_t n, int ncol, const double* y, int64_t nrow, int64_t ld,
                                  double* D, void* work, int64_t work_bytes, void* stream) {
  return dots_impl<double>(X, n, ncol, y, nrow, ld, D, work, work_bytes, stream);
}
extern "C" int mk_design_apply_f32(const float* base, int64_t nrow, int64_t n, int64_t ld, const double* X, int ncol,
                                   int c0, int nk, const double* coef, float* out, int64_t ld_out, void* stream) {
  return apply_impl<float>(base, nrow, n, ld, X, ncol, c0, nk, coef, out, ld_out, stream);
}
extern "C" int mk_design_apply_f64(const double* base, int64_t nrow, int64_t n, int64_t ld, const double* X,
                                   int ncol, int c0, int nk, const double* coef, double* out, int64_t ld_out,
                                   void* stream) {
  return apply_impl<double>(base, nrow, n, ld, X, ncol, c0, nk, coef, out, ld_out, stream);
}
