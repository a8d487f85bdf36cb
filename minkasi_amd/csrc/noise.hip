// Spectrum smoothing for NoiseSmoothedSVD setup (minkasi/mapmaking/noise.py:
// 674-678 with smooth_many_vecs, minkasi/tools/smooth.py:49-78).
//
// smooth_many_vecs computes DCT-I(DCT-I(P) * DCT-I(g)) / (2(n-1)) with g the
// r2r-normalised Gaussian.  Because DCT-I o DCT-I = 2(n-1) I, that equals the
// circular (period 2(n-1)) convolution of the even extensions of P and g,
// S_k = sum_{t in (-m, m]} g[|t|] P_ext(k - t), m = n-1.  The Gaussian
// underflows far from its centre, so the sum is evaluated directly over the
// taps the host passes (|t| up to ~13 sigma, or the whole period when the
// row is shorter), in FP64, with the input window staged in LDS.  Optionally
// the input is squared first (P = DCT(v.d)^2) and the output inverted with
// bin 0 set to zero (mywt = 1/S, mywt[:, 0] = 0).
#include "common.h"

namespace {

constexpr int kOut = 8;             // consecutive outputs per thread
constexpr int kThreads = 128;
constexpr int kChunk = kOut * kThreads;

// Window element w in LDS: one element of padding every 8 spreads the
// threads' windows, which start 8 apart, over the banks.
__host__ __device__ constexpr int wpos(int w) { return w + (w >> 3); }

// Bound by the FP64 unit.  A thread slides the taps over kOut outputs: 8 taps
// and 15 window values make 64 fused multiply-adds, so a product costs 1/8 LDS
// read (the taps are scalar) against one per product for an output per thread.
// Every output still sums its taps in ascending order.  215 x 90001, 553 taps:
// 739 us from 2457.
__global__ void __launch_bounds__(kThreads) smooth_kernel(const double* __restrict__ x, int64_t n, int64_t chunks,
                                                          const double* __restrict__ g, int t_lo, int t_hi, int flags,
                                                          double* __restrict__ out, float* __restrict__ out32) {
  extern __shared__ double win[];  // wpos(kChunk + t_hi - t_lo) elements
  const int64_t row = blockIdx.x / chunks;
  const int64_t k0 = (blockIdx.x % chunks) * kChunk;
  const int64_t m = n - 1;
  const double* xr = x + row * n;
  const int wlen = kChunk + t_hi - t_lo;
  // win[w] = P_ext(k0 - t_hi + w), P_ext even about 0 and about m.  Every
  // sample an output needs lies in [-m, 2m]; the rest of the last window is
  // any sample.
  for (int w = threadIdx.x; w < wlen; w += kThreads) {
    int64_t i = k0 - t_hi + w;
    if (i < 0) i = -i;
    if (i > m) i = 2 * m - i;
    i = max((int64_t)0, min(i, m));
    const double v = xr[i];
    win[wpos(w)] = (flags & 1) ? v * v : v;
  }
  __syncthreads();
  // S_k = sum_t g[|t|] P(k - t): P(k - t) = win[c + t_hi - t]
  const int c0 = threadIdx.x * kOut;
  double acc[kOut];
#pragma unroll
  for (int r = 0; r < kOut; r++) acc[r] = 0.0;
  int t = t_lo, top = c0 + t_hi - t_lo;  // output r reads window element top + r at tap t
  double a[kOut], b[kOut];               // elements top .. top + 7 and top - 8 .. top - 1
  if (t + kOut <= t_hi + 1) {
#pragma unroll
    for (int r = 0; r < kOut; r++) a[r] = win[wpos(top + r)];
  }
  for (; t + kOut <= t_hi + 1; t += kOut, top -= kOut) {
#pragma unroll
    for (int r = 0; r < kOut; r++) b[r] = win[wpos(max(top - kOut + r, 0))];  // -1 only after the last tap
#pragma unroll
    for (int q = 0; q < kOut; q++) {
      const double gt = g[t + q < 0 ? -(t + q) : t + q];
#pragma unroll
      for (int r = 0; r < kOut; r++) acc[r] = fma(gt, r >= q ? a[r - q] : b[kOut + r - q], acc[r]);
    }
#pragma unroll
    for (int r = 0; r < kOut; r++) a[r] = b[r];
  }
  for (; t <= t_hi; t++, top--) {
    const double gt = g[t < 0 ? -t : t];
#pragma unroll
    for (int r = 0; r < kOut; r++) acc[r] = fma(gt, win[wpos(top + r)], acc[r]);
  }
  __syncthreads();  // the window is done with: the sums go out through it in row order
#pragma unroll
  for (int r = 0; r < kOut; r++) win[wpos(c0 + r)] = acc[r];
  __syncthreads();
  for (int c = threadIdx.x; c < kChunk; c += kThreads) {
    const int64_t k = k0 + c;
    if (k >= n) break;
    double s = win[wpos(c)];
    if (flags & 2) s = (k == 0) ? 0.0 : 1.0 / s;
    out[row * n + k] = s;
    if (out32) out32[row * n + k] = (float)s;
  }
}

}  // namespace

extern "C" int mk_smooth_rows_f64(const double* x, double* out, float* out32, int64_t nrow, int64_t n,
                                  const double* g, int32_t t_lo, int32_t t_hi, int32_t flags, void* stream) {
  MK_REQUIRE(nrow >= 0 && n >= 2, MK_ERR_ARG, "need n >= 2");
  if (nrow == 0) return MK_OK;
  MK_REQUIRE(x && out && g, MK_ERR_ARG, "null argument");
  MK_REQUIRE(t_lo <= 0 && t_hi >= 0 && t_hi - t_lo < 2 * (n - 1) + 1 && -t_lo <= n - 1 && t_hi <= n - 1,
             MK_ERR_ARG, "taps must satisfy -(n-1) <= t_lo <= 0 <= t_hi <= n-1");
  MK_REQUIRE(t_hi - t_lo <= 16384, MK_ERR_ARG, "too many taps");
  MK_REQUIRE(x != out, MK_ERR_ARG, "smoothing cannot run in place");
  int64_t chunks = mk::cdiv(n, kChunk);
  size_t lds = (size_t)(wpos(kChunk + t_hi - t_lo) + 1) * sizeof(double);  // at most 153 KB
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(smooth_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                            160 * 1024);
  (void)hipGetLastError();
  smooth_kernel<<<(unsigned)(nrow * chunks), kThreads, lds, mk::as_stream(stream)>>>(x, n, chunks, g, t_lo, t_hi, flags,
                                                                               out, out32);
  return mk::check_launch("smooth_kernel");
}
