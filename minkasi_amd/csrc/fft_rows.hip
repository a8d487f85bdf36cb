// Row pass of the 2^11-point-row FFT engine and its twiddle tables.
//
// 256 threads transform two rows of 2^11 points, 16 points per thread, in
// three stages of radix 16, 16 and 8: the first reads global memory straight
// into registers, the other two exchange through LDS.  The inverse mirrors
// it (8, 16, 16), so forward, spectral step and inverse need four LDS
// exchanges.  In the last forward stage one thread holds butterfly k of one
// row and the butterfly that carries the partner frequencies P - k of the
// other (rows k1 and Q1 - k1, or one self-paired row), so the spectral step
// and the first inverse stage stay in its registers.
//
// The four-step twiddle w_P^(k1 j2) costs no extra pass: with
// j2 = j + 128 r the stages see it as w_(16 Q1)^(k1 r) on the inputs and as
// factors w_(256 Q1)^(k1 r), w_P^(k1 r) of the stage twiddles, all uniform
// over a row (scalar loads from a table per column count).
//
// Bound: HBM; per point of the filter 8 B in, 8 B of spectrum and 8 B out
// (215 rows of 100003 samples, 22e6 points: 0.53 GB in 122 us, 4.3 TB/s; the
// eleven-exchange pass over rows 1.5 times as long that this replaces took
// 262 us).  Three waves per SIMD without spills beat four with 12 spilled
// registers (125 against 160 us); loading the spectrum before the second
// stage instead of after it gains 2 % in FP32 and costs 15 % in FP64 (spills).
#include "fft_engine.h"

namespace mkfft {
namespace {

constexpr int kRowPad = kRowLen + kRowLen / 16 + 1;  // element e of a row lies at e + e/16: no bank conflicts

template <typename TS>
struct alignas(2 * sizeof(TS)) Spec2 {
  TS h, g;
};

template <typename TS>
__device__ __forceinline__ Spec2<TS> load_spec(gptr<const Spec2<TS>> p) {
  typedef TS V2 __attribute__((ext_vector_type(2)));
  const V2 v = *(gptr<const V2>)p;
  return {v.x, v.y};
}

// One frequency pair of the filter (k, P - k), C = C_k, Cq = C_(P-k) of the
// packed transform, wp = -i w_L^k, in place.  With S+- = u +- wp d
// (u = C + conj Cq, d = C - conj Cq: twice the real transform at k and the
// conjugate of twice it at P - k), the convolution's spectrum is
//   Y = H S + G phi conj(S),
// H and G the (real) spectra of the kernel and of the kernel reversed about
// m/2, phi = 1 (m even) or conj(w_L^k) (m odd, the reversal's centre lies
// half a sample off the grid); phi at P - k is conj(phi) (m even) or
// -w_L^k.  Four times the packed result; the column pass scales it.
template <typename T, typename TS>
__device__ __forceinline__ void spectral_pair(cx<T>& C, cx<T>& Cq, cx<T> wp, Spec2<TS> a, Spec2<TS> aq, bool odd) {
  const cx<T> u = {C.re + Cq.re, C.im - Cq.im}, d = {C.re - Cq.re, C.im + Cq.im};
  const cx<T> wd = cmul(wp, d);
  const cx<T> Sp = cadd(u, wd), Sm = csub(u, wd);
  const T h = (T)a.h, g = (T)a.g, hq = (T)aq.h, gq = (T)aq.g;
  cx<T> Y, Yq;  // Yq: the conjugate of the value at P - k
  if (!odd) {
    Y = {(h + g) * Sp.re, (h - g) * Sp.im};
    Yq = {(hq + gq) * Sm.re, (hq - gq) * Sm.im};
  } else {
    // phi = conj(w) = conj(i wp) = -i conj(wp)
    const cx<T> phi = {-wp.im, -wp.re};
    const cx<T> tp = cmul(phi, cconj(Sp)), tm = cmul(phi, cconj(Sm));
    Y = {h * Sp.re + g * tp.re, h * Sp.im + g * tp.im};
    Yq = {hq * Sm.re - gq * tm.re, hq * Sm.im - gq * tm.im};
  }
  const cx<T> s = cadd(Y, Yq), e = cmul(cconj(wp), csub(Y, Yq));
  C = cadd(s, e);
  Cq = cconj(csub(s, e));
}

// The real transform's values at k and P - k (real for a symmetric kernel).
template <typename T>
__device__ __forceinline__ void real_pair(cx<T> C, cx<T> Cq, cx<T> wp, T* ak, T* aq) {
  const cx<T> u = {C.re + Cq.re, C.im - Cq.im}, d = {C.re - Cq.re, C.im + Cq.im};
  const T r = wp.re * d.re - wp.im * d.im;
  *ak = T(0.5) * (u.re + r);
  *aq = T(0.5) * (u.re - r);
}

template <typename T, typename TS, int MODE>
__global__ void __launch_bounds__(kRowThreads, sizeof(T) == 4 ? 3 : 2)
    rows_kernel(const Seg* __restrict__ segs, int nseg, cx<T>* __restrict__ tbuf, const cx<T>* __restrict__ common,
                int comp) {
  extern __shared__ unsigned char smem_raw[];
  cx<T>* X = reinterpret_cast<cx<T>*>(smem_raw);  // [2][kRowPad]
  const Seg& sg = segs[find_seg(segs, nseg, blockIdx.x, 2)];
  const int local = (int)((int64_t)blockIdx.x - sg.base2);
  const int row = local / sg.per2, g = local - row * sg.per2;
  const int Q = sg.q1, P = Q << kRowL2;
  constexpr bool PAIRED = MODE == kFilter || MODE == kFSpec;
  // rows k1 of this workgroup; `single`: there is no second one, and its
  // threads work on a copy of the first that is never stored
  int kA, kB;
  bool single;
  if constexpr (PAIRED) {
    kA = g;
    single = g == 0 && (Q & 1);
    kB = g == 0 ? (single ? 0 : Q / 2) : Q - g;
  } else {
    kA = 2 * g;
    single = 2 * g + 1 >= Q;
    kB = single ? kA : kA + 1;
  }
  const int tid = threadIdx.x;
  const int rsel = __builtin_amdgcn_readfirstlane(tid >> 7);  // this wave's row in the radix-16 stages
  const int j = tid & 127;
  const int kr = rsel ? kB : kA;
  cx<T>* trow = tbuf + sg.t_off + (int64_t)row * sg.t_stride;
  const cx<T>* rt = common + sg.tw_off;
  const cx<T>* rtr = rt + kr * kRowTw;
  cx<T>* Xr = X + rsel * kRowPad;
  const int jp = j + (j >> 4), jq = (j >> 4) * 272 + (j & 15);
  cx<T>* io = trow + (int64_t)kr * kRowLen + j;

  cx<T> v[16];
#pragma unroll
  for (int r = 0; r < 16; r++) v[r] = io[128 * r];
#pragma unroll
  for (int r = 1; r < 16; r++) v[r] = cmul(v[r], rtr[r]);
  dft_small<T, false, 16>(v);
#pragma unroll
  for (int r = 0; r < 16; r++) Xr[17 * j + r] = v[r];
  __syncthreads();

  // last stage: butterfly ka of row sa and kb of row sb, elements r at
  // k2 = ka + 256 r; the partner of (sa, ka, r) is (sb, kb, 7 - r)
  int sa = 0, sb = 1, ka = tid, kb = 255 - tid;
  bool self0 = false;
  if (PAIRED && g == 0) {
    sa = sb = rsel;
    ka = j;
    kb = rsel ? 255 - j : (256 - j) & 255;
    if (tid == 0) {  // row k1 = 0: k2 = 0 and 128 pair within their own butterflies
      self0 = true;
      kb = 128;
    }
  }
  const int k1a = sa ? kB : kA, k1b = sb ? kB : kA;
  Spec2<TS> ha[8], hb[8];
  TS hP{}, gP{};
  auto load_spectrum = [&]() {
    if constexpr (MODE == kFilter) {
      const gptr<const Spec2<TS>> sp = as_global<const Spec2<TS>>(sg.s_ptr) + (int64_t)row * (sg.s_stride >> 1);
#pragma unroll
      for (int r = 0; r < 8; r++) {
        ha[r] = load_spec(sp + k1a * kRowLen + ka + 256 * r);
        hb[r] = load_spec(sp + k1b * kRowLen + kb + 256 * r);
      }
      if (self0) {
        hP = sp[P].h;
        gP = sp[P].g;
      }
    } else if constexpr (MODE == kBlue) {
      const gptr<const cx<T>> V = as_global<const cx<T>>(sg.s_ptr);
#pragma unroll
      for (int r = 0; r < 8; r++) {
        ha[r] = load_spec((gptr<const Spec2<TS>>)V + k1a * kRowLen + ka + 256 * r);
        hb[r] = load_spec((gptr<const Spec2<TS>>)V + k1b * kRowLen + kb + 256 * r);
      }
    }
  };
  // in flight over the second stage; FP64, whose registers would spill, loads
  // after it
  if constexpr (sizeof(T) == 4) load_spectrum();

#pragma unroll
  for (int r = 0; r < 16; r++) v[r] = Xr[jp + 136 * r];
#pragma unroll
  for (int r = 1; r < 16; r++) v[r] = cmul(v[r], cmul(common[r * 16 + (j & 15)], rtr[16 + r]));
  dft_small<T, false, 16>(v);
  if constexpr (sizeof(T) == 8) load_spectrum();
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; r++) Xr[jq + 17 * r] = v[r];
  __syncthreads();

  cx<T>* Xa = X + sa * kRowPad + ka + (ka >> 4);
  cx<T>* Xb = X + sb * kRowPad + kb + (kb >> 4);
  const cx<T>* rta = rt + k1a * kRowTw;
  const cx<T>* rtb = rt + k1b * kRowTw;
  cx<T> a[8], b[8], ta[8], tb[8];
#pragma unroll
  for (int r = 0; r < 8; r++) {
    a[r] = Xa[272 * r];
    b[r] = Xb[272 * r];
  }
#pragma unroll
  for (int r = 1; r < 8; r++) {
    ta[r] = cmul(common[256 + r * 256 + ka], rta[32 + r]);
    tb[r] = cmul(common[256 + r * 256 + kb], rtb[32 + r]);
    a[r] = cmul(a[r], ta[r]);
    b[r] = cmul(b[r], tb[r]);
  }
  dft_small<T, false, 8>(a);
  dft_small<T, false, 8>(b);

  if constexpr (MODE == kBSpec) {
    const gptr<cx<T>> V = as_global<cx<T>>(sg.s_ptr);
#pragma unroll
    for (int r = 0; r < 8; r++) {
      const gptr<cx<T>> va = V + k1a * kRowLen + ka + 256 * r, vb = V + k1b * kRowLen + kb + 256 * r;
      va->re = a[r].re;
      va->im = a[r].im;
      if (!single) {
        vb->re = b[r].re;
        vb->im = b[r].im;
      }
    }
    return;
  }
  if constexpr (MODE == kBlue) {
#pragma unroll
    for (int r = 0; r < 8; r++) {
      a[r] = cmul(a[r], cx<T>{(T)ha[r].h, (T)ha[r].g});
      b[r] = cmul(b[r], cx<T>{(T)hb[r].h, (T)hb[r].g});
    }
  } else {
    // wp = -i w_2P^k at k = k1 + Q (k2 + 256 r): w_2P^k1 w_4096^k2 w_16^r
    const cx<T> w0 = cmul(rta[40], common[2304 + ka]);
    const cx<T> wp0 = {w0.im, -w0.re};
    if constexpr (MODE == kFSpec) {
      if (single && rsel) return;
      const gptr<TS> srow = as_global<TS>(sg.s_ptr) + (int64_t)row * sg.s_stride + comp;
      auto put = [&](int k1, int k2, T val) { srow[2 * ((int64_t)k1 * kRowLen + k2)] = (TS)val; };
      if (!self0) {
#pragma unroll
        for (int r = 0; r < 8; r++) {
          T x, y;
          real_pair(a[r], b[7 - r], mul_w16<T, false>(wp0, r), &x, &y);
          put(k1a, ka + 256 * r, x);
          put(k1b, kb + 256 * (7 - r), y);
        }
      } else {
        T x, y;
        put(0, 0, a[0].re + a[0].im);
        srow[2 * (int64_t)P] = (TS)(a[0].re - a[0].im);
#pragma unroll
        for (int r = 1; r <= 4; r++) {
          real_pair(a[r], a[8 - r], mul_w16<T, false>(wp0, r), &x, &y);
          put(0, 256 * r, x);
          if (r < 4) put(0, 256 * (8 - r), y);
        }
        const cx<T> w1 = cmul(rta[40], common[2304 + 128]);
        const cx<T> wp1 = {w1.im, -w1.re};
#pragma unroll
        for (int r = 0; r < 4; r++) {
          real_pair(b[r], b[7 - r], mul_w16<T, false>(wp1, r), &x, &y);
          put(0, 128 + 256 * r, x);
          put(0, 128 + 256 * (7 - r), y);
        }
      }
      return;
    } else {
      const bool odd = ((sg.n - 1) & 1) != 0;
      if (!self0) {
#pragma unroll
        for (int r = 0; r < 8; r++)
          spectral_pair<T, TS>(a[r], b[7 - r], mul_w16<T, false>(wp0, r), ha[r], hb[7 - r], odd);
      } else {
        const T a0 = a[0].re + a[0].im, aP = a[0].re - a[0].im;
        const T y0 = ((T)ha[0].h + (T)ha[0].g) * a0;
        const T yP = (odd ? (T)hP - (T)gP : (T)hP + (T)gP) * aP;
        a[0] = {T(2) * (y0 + yP), T(2) * (y0 - yP)};
#pragma unroll
        for (int r = 1; r < 4; r++)
          spectral_pair<T, TS>(a[r], a[8 - r], mul_w16<T, false>(wp0, r), ha[r], ha[8 - r], odd);
        cx<T> dup = a[4];  // k = P/2 is its own partner
        spectral_pair<T, TS>(a[4], dup, mul_w16<T, false>(wp0, 4), ha[4], ha[4], odd);
        const cx<T> w1 = cmul(rta[40], common[2304 + 128]);
        const cx<T> wp1 = {w1.im, -w1.re};
#pragma unroll
        for (int r = 0; r < 4; r++)
          spectral_pair<T, TS>(b[r], b[7 - r], mul_w16<T, false>(wp1, r), hb[r], hb[7 - r], odd);
      }
    }
  }

  // inverse: 8, 16, 16
  dft_small<T, true, 8>(a);
  dft_small<T, true, 8>(b);
  Xa[0] = a[0];
  Xb[0] = b[0];
#pragma unroll
  for (int r = 1; r < 8; r++) {
    Xa[272 * r] = cmul(a[r], cconj(ta[r]));
    Xb[272 * r] = cmul(b[r], cconj(tb[r]));
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; r++) v[r] = Xr[jq + 17 * r];
  dft_small<T, true, 16>(v);
#pragma unroll
  for (int r = 1; r < 16; r++) v[r] = cmul(v[r], cconj(cmul(common[r * 16 + (j & 15)], rtr[16 + r])));
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; r++) Xr[jp + 136 * r] = v[r];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; r++) v[r] = Xr[17 * j + r];
  dft_small<T, true, 16>(v);
  if (single && rsel) return;
  io[0] = v[0];
#pragma unroll
  for (int r = 1; r < 16; r++) io[128 * r] = cmul(v[r], cconj(rtr[r]));
}

// Tables of one column count (and the common ones), computed in FP64.
template <typename T>
__global__ void col_tables_kernel(int q, cx<T>* __restrict__ common, cx<T>* __restrict__ tab) {
  const int nc = common ? kTwCommon : 0, total = nc + (int)(q * (kRowTw + 1));
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < total; e += gridDim.x * blockDim.x) {
    int64_t num, den;  // exp(-2 pi i num / den)
    cx<T>* out;
    if (e < nc) {
      out = common + e;
      if (e < 256) { num = (e & 15) * (e >> 4); den = 256; }
      else if (e < 2304) { num = (e & 255) * ((e - 256) >> 8); den = 2048; }
      else { num = e - 2304; den = 4096; }
    } else {
      const int t = e - nc;
      out = tab + t;
      if (t < q * kRowTw) {
        const int k1 = t / kRowTw, f = t % kRowTw;
        if (f < 16) { num = (int64_t)k1 * f; den = 16 * (int64_t)q; }
        else if (f < 32) { num = (int64_t)k1 * (f - 16); den = 256 * (int64_t)q; }
        else if (f < 40) { num = (int64_t)k1 * (f - 32); den = 2048 * (int64_t)q; }
        else { num = k1; den = 4096 * (int64_t)q; }
      } else {
        num = t - q * kRowTw;
        den = q;
      }
    }
    double s, c;
    sincospi(-2.0 * (double)(num % den) / (double)den, &s, &c);
    *out = {(T)c, (T)s};
  }
}

// The end modes' phases of rows of n samples on q columns: exp(i pi t / m),
// t = i + c0 for i < 2^12, then t = 2^12 j1 (less 2P in the upper half of the
// time rows) for j1 < q.
template <typename T>
__global__ void end_phase_kernel(cx<T>* __restrict__ out, int64_t n, int q) {
  const int64_t m = n - 1, c0 = (m + 1) >> 1;
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < 2 * kRowLen + q; e += gridDim.x * blockDim.x) {
    const int j1 = e - 2 * kRowLen;
    const int64_t t = j1 < 0 ? e + c0 : 2 * (int64_t)kRowLen * (j1 - (2 * j1 >= q ? q : 0));
    double s, c;
    sincospi((double)t / (double)m, &s, &c);
    out[e] = {(T)c, (T)s};
  }
}

// Per row of h = C W the first two values of C h = 2m W: the filter's
// eigenvalues for the constant and for cos(pi j / m), stored behind the
// row's spectra.  One workgroup per row, fixed-order FP64 sums.
template <typename TS>
__global__ void __launch_bounds__(1024) end_modes_kernel(const Seg* __restrict__ segs, int nseg,
                                                        const double* __restrict__ h_all) {
  __shared__ double sh[2][1024];
  int64_t g = blockIdx.x;
  int i = 0;
  while (g >= segs[i].rows) g -= segs[i++].rows;
  const Seg& sg = segs[i];
  const double* h = h_all + sg.in_off + g * sg.in_stride;
  const int m = sg.n - 1;
  double e0 = 0.0, e1 = 0.0;
  for (int j = threadIdx.x; j <= m; j += 1024) {
    const double v = h[j] * (j == 0 || j == m ? 1.0 : 2.0);
    e0 += v;
    e1 += v * cospi((double)j / (double)m);
  }
  sh[0][threadIdx.x] = e0;
  sh[1][threadIdx.x] = e1;
  __syncthreads();
  for (int t = 512; t > 0; t >>= 1) {
    if ((int)threadIdx.x < t) {
      sh[0][threadIdx.x] += sh[0][threadIdx.x + t];
      sh[1][threadIdx.x] += sh[1][threadIdx.x + t];
    }
    __syncthreads();
  }
  if (threadIdx.x < 2)
    (as_global<TS>(sg.s_ptr) + g * sg.s_stride)[2 * (sg.t_stride + 1) + threadIdx.x] = (TS)sh[threadIdx.x][0];
}

// exp(-i pi j^2 / N), N = 2(n-1), for j < n.
__global__ void chirp_kernel(cx<double>* __restrict__ out, int64_t n) {
  const int64_t N = 2 * (n - 1);
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (int64_t)gridDim.x * blockDim.x)
    out[j] = expmi<double>((j * j) % (2 * N), N);
}

template <typename T, typename TS, int MODE>
void launch_rows_mode(const Seg* segs, int nseg, int64_t nblk, cx<T>* tbuf, const cx<T>* common, int comp,
                      hipStream_t st) {
  constexpr int lds = 2 * kRowPad * (int)sizeof(cx<T>);
  rows_kernel<T, TS, MODE><<<(unsigned)nblk, kRowThreads, lds, st>>>(segs, nseg, tbuf, common, comp);
}

template <typename TS, int MODE>
void allow_lds64() {
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(rows_kernel<double, TS, MODE>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, 2 * kRowPad * (int)sizeof(cx<double>));
}

}  // namespace

void allow_rows_lds() {
  allow_lds64<double, kFilter>();
  allow_lds64<double, kFSpec>();
  allow_lds64<float, kFSpec>();
  allow_lds64<double, kBlue>();
  allow_lds64<double, kBSpec>();
}

template <>
void launch_rows<float>(int mode, const Seg* segs, int nseg, int64_t nblk, cx<float>* tbuf, const cx<float>* common,
                        int comp, bool, hipStream_t st) {
  (void)mode;  // FP32 rows run the filter only
  launch_rows_mode<float, float, kFilter>(segs, nseg, nblk, tbuf, common, comp, st);
}
template <>
void launch_rows<double>(int mode, const Seg* segs, int nseg, int64_t nblk, cx<double>* tbuf,
                         const cx<double>* common, int comp, bool spec32, hipStream_t st) {
  if (mode == kFilter) launch_rows_mode<double, double, kFilter>(segs, nseg, nblk, tbuf, common, comp, st);
  else if (mode == kFSpec && spec32)
    launch_rows_mode<double, float, kFSpec>(segs, nseg, nblk, tbuf, common, comp, st);
  else if (mode == kFSpec) launch_rows_mode<double, double, kFSpec>(segs, nseg, nblk, tbuf, common, comp, st);
  else if (mode == kBlue) launch_rows_mode<double, double, kBlue>(segs, nseg, nblk, tbuf, common, comp, st);
  else launch_rows_mode<double, double, kBSpec>(segs, nseg, nblk, tbuf, common, comp, st);
}
template <typename T>
void launch_col_tables(int q, cx<T>* common, cx<T>* tab, hipStream_t st) {
  const int64_t total = (common ? kTwCommon : 0) + q1_table_elems(q);
  col_tables_kernel<T><<<mk::grid_for(total, 256), 256, 0, st>>>(q, common, tab);
}
template void launch_col_tables<float>(int, cx<float>*, cx<float>*, hipStream_t);
template void launch_col_tables<double>(int, cx<double>*, cx<double>*, hipStream_t);
template <typename T>
void launch_end_phases(cx<T>* out, int64_t n, int q, hipStream_t st) {
  end_phase_kernel<T><<<mk::grid_for(2 * kRowLen + q, 256), 256, 0, st>>>(out, n, q);
}
template void launch_end_phases<float>(cx<float>*, int64_t, int, hipStream_t);
template void launch_end_phases<double>(cx<double>*, int64_t, int, hipStream_t);
void launch_end_modes(const Seg* segs, int nseg, int64_t rows, const double* h, bool spec32, hipStream_t st) {
  if (spec32) end_modes_kernel<float><<<(unsigned)rows, 1024, 0, st>>>(segs, nseg, h);
  else end_modes_kernel<double><<<(unsigned)rows, 1024, 0, st>>>(segs, nseg, h);
}
void launch_chirp(cx<double>* chirp, int64_t n, hipStream_t st) {
  chirp_kernel<<<mk::grid_for(n, 256), 256, 0, st>>>(chirp, n);
}

}  // namespace mkfft
