// Batched four-step FFT engine and the two transforms built on it.
//
// NoiseSmoothedSVD.apply_noise (minkasi/mapmaking/noise.py:704-711) applies,
// per rotated detector mode y (length n), y'' = C W C y where C is the
// unnormalised DCT-I (FFTW REDFT00, minkasi/lib/mkfftw.c:174-212;
// scipy.fft.dct type 1, minkasi/tools/py_fft.py:239) and W = mywt.  With
// m = n-1 and N = 2m, C W C y = (even extension of y) circularly convolved
// (period N) with h = C W (because C C = N I).  The engine evaluates that
// circular convolution exactly through real FFTs, for any n (no Bluestein,
// no smooth-length requirement), and fuses the forward transform, the weight
// multiply and the inverse transform.  Two forms:
//
//  2^11-row path (FP32 and FP64 rows of about 1400 to 2^19 samples;
//  fft_cols.h, fft_rows.hip).  With the end samples halved, the output is
//  sum_j y_j [h(k-j) + h(k+j)], a Toeplitz product plus one with a kernel
//  reversed about m/2 (h(k+j) = h(k - (m-j) + m)): as spectra
//  H Y + G phi conj(Y) with Y one real transform of L >= 2m+1 points, H and
//  G the real spectra of h(|t|) and h(m-|t|), |t| <= m, and phi the phase of
//  the reversal's centre.  L = 2^12 q1, q1 the smallest of 41 counts that
//  split into two radices up to 16.
//
//  General path (shorter and longer rows).  The even extension on [-m, 2m]
//  through L >= 3m+1 points with one real spectrum; the outputs needed are
//  the window [m, 2m]; L a power of two.
//
// Stand-alone DCT-I (fft_r2r, minkasi/tools/fft.py:290-344) uses Bluestein's
// chirp-z algorithm (Bluestein 1970; Rabiner, Schafer & Rader 1969) on the
// same engines: Y_k = Re(chi_k sum_j c_j x_j chi_j conj(chi_{k-j})) with
// chi_j = exp(-i pi j^2 / N), c_j = 1 at j = 0, m and 2 otherwise, the
// convolution evaluated with a complex FFT of P >= 2m+1 points (FP64: 2^11 q1,
// else a power of two).
//
// General path's four-step layout (P = P1*P2 complex points, j = P2*j1 + j2,
// k = k1 + P1*k2):
//   K1: column FFTs of length P1 (one workgroup = cw adjacent columns, so
//       global reads are contiguous runs), twiddle w_P^(j2*k1), store T[k1][j2].
//   K2: row FFTs of length P2 (rows k1 and P1-k1 together, which is where the
//       real-FFT unpacking partner C_(P-k) lives), pointwise spectral work,
//       inverse row FFTs, conjugate twiddle, store back.
//   K3: inverse column FFTs of length P1, 1/P scale, write the wanted outputs.
// Every LDS sub-FFT is a Stockham pass sequence (radix 8, then 4 or 2) with a
// stage-ordered twiddle table.
// Each launch covers every row of every segment (TOD) in the batch through
// a work list.
#include "fft_engine.h"

#include <algorithm>
#include <cstdlib>
#include <mutex>
#include <vector>

using namespace mkfft;

namespace {

// exp(-i*pi*num*inv_den) with 1/inv_den a power of two and num < 2^24, so
// -num * inv_den is exact in T.
template <typename T>
__device__ __forceinline__ cx<T> expmi2(int64_t num, T inv_den) {
  T s, c;
  sincospi_t(-(T)num * inv_den, &s, &c);
  return {c, s};
}

constexpr int kThreads = 512;                  // threads per FFT workgroup
constexpr int kMaxWG = 4096;                   // complex points per workgroup in an LDS FFT (8 per thread)
constexpr int kMaxLds = 144 * 1024;            // dynamic LDS budget per workgroup (gfx950 has 160 KB)

// LDS rows are padded: element e of a row lives at e + e/16 (measured best of
// e/8, e/16, e/32 and none on gfx950) and rows are
// row_stride(len) apart (odd), so the strided Stockham writes of the early
// radix-8 stages, the row-parallel writes of K1/K3 and the unit-stride reads
// all map to distinct banks.
#ifndef MK_FFT_PAD_SHIFT
#define MK_FFT_PAD_SHIFT 4
#endif
constexpr __host__ __device__ __forceinline__ int pad8(int e) { return e + (e >> MK_FFT_PAD_SHIFT); }
// Odd, so that rows read in parallel fall in different banks (for a power of
// two len this is len + len/16 + 1).
constexpr __host__ __device__ __forceinline__ int row_stride(int len) { return (len + (len >> MK_FFT_PAD_SHIFT)) | 1; }

// One radix-R Stockham stage over nrows padded rows of length 2^l2len.
// Every thread loads all of its butterflies' inputs, the workgroup
// synchronises, then the outputs are written in place.
// tw: this stage's twiddles, tw[(r-1)*Ns + k] = exp(-2 pi i k r / (R Ns)),
// so the lanes of a wave (consecutive k) read consecutive words.
template <typename T, bool INV, int LR>
__device__ __forceinline__ void fft_stage(cx<T>* buf, const cx<T>* tw, int l2len, int nrows, int rs, int Ns,
                                          int lns) {
  constexpr int R = 1 << LR;
  constexpr int NB = kMaxWG / R / kThreads;
  const int lq = l2len - LR, q = 1 << lq;
  const int nbf = nrows << lq;
  cx<T> v[NB][R];
#pragma unroll
  for (int u = 0; u < NB; u++) {
    int bf = threadIdx.x + u * kThreads;
    if (bf < nbf) {
      int row = bf >> lq, j = bf & (q - 1), k = j & (Ns - 1);
      const cx<T>* base = buf + row * rs;
#pragma unroll
      for (int r = 0; r < R; r++) v[u][r] = base[pad8(j + r * q)];
      if (lns > 0) {
#pragma unroll
        for (int r = 1; r < R; r++) {
          cx<T> w = tw[(r - 1) * Ns + k];
          if (INV) w = cconj(w);
          v[u][r] = cmul(v[u][r], w);
        }
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NB; u++) {
    int bf = threadIdx.x + u * kThreads;
    if (bf < nbf) {
      int row = bf >> lq, j = bf & (q - 1), k = j & (Ns - 1);
      if (LR == 3) dft8<T, INV>(v[u]);
      else if (LR == 2) dft4v<T, INV>(v[u]);
      else dft2<T, INV>(v[u]);
      cx<T>* base = buf + row * rs;
      int idx = ((j >> lns) << (lns + LR)) + k;
#pragma unroll
      for (int r = 0; r < R; r++) base[pad8(idx + r * Ns)] = v[u][r];
    }
  }
  __syncthreads();
}

// Radix of the stage that follows `rem` remaining levels: 8 while three or
// more levels remain, then 4 or 2.
__host__ __device__ __forceinline__ int stage_lr(int rem) { return rem >= 3 ? 3 : rem; }

// In-place FFT of nrows padded rows (row stride rs) of length 2^l2len,
// nrows * 2^l2len <= kMaxWG; tw = stage-ordered table (fill_stage_table).
template <typename T, bool INV>
__device__ void lds_fft(cx<T>* buf, const cx<T>* tw, int l2len, int nrows, int rs) {
  int Ns = 1, lns = 0, rem = l2len, off = 0;
  while (rem > 0) {
    const int lr = stage_lr(rem);
    if (lr == 3) fft_stage<T, INV, 3>(buf, tw + off, l2len, nrows, rs, Ns, lns);
    else if (lr == 2) fft_stage<T, INV, 2>(buf, tw + off, l2len, nrows, rs, Ns, lns);
    else fft_stage<T, INV, 1>(buf, tw + off, l2len, nrows, rs, Ns, lns);
    off += ((1 << lr) - 1) * Ns;
    Ns <<= lr; lns += lr; rem -= lr;
  }
}

// Twiddles of every stage of a length-2^l2len FFT, stage after stage:
// entry (r-1)*Ns + k of a stage is exp(-2 pi i k r / (R Ns)); 2^l2len - 1
// entries in all.
template <typename T>
__device__ void fill_stage_table(cx<T>* tab, int l2len) {
  const T inv = T(1) / (T)(1 << l2len);
  int Ns = 1, rem = l2len, off = 0;
  while (rem > 0) {
    const int lr = stage_lr(rem), R = 1 << lr;
    const int cnt = (R - 1) * Ns;
    const int mul = 1 << (l2len - lr - (l2len - rem));  // len / (R Ns)
    for (int e = threadIdx.x; e < cnt; e += kThreads) {
      int r = e / Ns + 1, k = e - (r - 1) * Ns;
      tab[off + e] = expmi2<T>(2 * (int64_t)k * r * mul, inv);
    }
    off += cnt;
    Ns <<= lr; rem -= lr;
  }
}

// exp(-2 pi i a / P) for 0 <= a < P, P = 2^lP <= 2^23.
template <typename T>
__device__ __forceinline__ cx<T> twiddle_P(int64_t a, T invP) { return expmi2<T>(2 * a, invP); }

// ---- K1: column FFTs -------------------------------------------------------
// LDS: cw padded rows of length P1 (one per matrix column j2), then the P1
// twiddle table and the P2 table exp(-2 pi i j/P) for the four-step twiddle.
template <typename T, typename TIn, int MODE>
__global__ void __launch_bounds__(kThreads, sizeof(T) == 4 ? 4 : 1) k1_kernel(const Seg* __restrict__ segs, int nseg,
                                                      const TIn* __restrict__ in, cx<T>* __restrict__ tbuf) {
  extern __shared__ unsigned char smem_raw[];
  const int s = find_seg(segs, nseg, blockIdx.x, 1);
  const Seg sg = segs[s];
  const int64_t local = (int64_t)blockIdx.x - sg.base1;
  const int row = (int)(local / sg.per1), jb = (int)(local % sg.per1);
  const int l1 = sg.l1, l2 = sg.l2, P1 = sg.p1, P2 = 1 << l2, cw = sg.cw;
  const int lcw = 31 - __clz(cw);
  const int rs = row_stride(P1);
  const int64_t P = (int64_t)P1 * P2;
  const int64_t m = sg.n - 1, N = 2 * m;
  cx<T>* buf = reinterpret_cast<cx<T>*>(smem_raw);  // [cw][rs]
  cx<T>* tw = buf + cw * rs;                          // [P1] stage table
  const TIn* x = in + sg.in_off + (int64_t)row * sg.in_stride;
  const int j2_0 = jb * cw;
  fill_stage_table<T>(tw, l1);
  constexpr int UNR = 8;  // loads in flight per thread
  if (MODE == kFilter || MODE == kFSpec) {
    // real input packed two per complex point: a_(2j), a_(2j+1)
    const int64_t L = 2 * P;
    const int total = P1 * cw * 2;
    for (int base = threadIdx.x; base < total; base += kThreads * UNR) {
      T val[UNR];
#pragma unroll
      for (int u = 0; u < UNR; u++) {
        int idx = base + u * kThreads;
        val[u] = T(0);
        if (idx < total) {
          int j1 = idx >> (lcw + 1), w = idx & (2 * cw - 1);
          int64_t i = 2 * ((int64_t)P2 * j1 + j2_0) + w;  // a-index
          if (MODE == kFilter) {
            if (i <= 3 * m) {
              int64_t t = i - m;
              int64_t src = t < 0 ? -t : (t <= m ? t : 2 * m - t);
              val[u] = (T)x[src];
            }
          } else {
            // symmetric embedding of h (rows of DCT-I(W)): b_i = h_i (i < m),
            // h_m/2 at i = m and L-m, h_(L-i) for L-m < i < L
            if (i < m) val[u] = (T)x[i];
            else if (i == m || i == L - m) val[u] = (T)x[m] * T(0.5);
            else if (i > L - m) val[u] = (T)x[L - i];
          }
        }
      }
#pragma unroll
      for (int u = 0; u < UNR; u++) {
        int idx = base + u * kThreads;
        if (idx < total) {
          int j1 = idx >> (lcw + 1), w = idx & (2 * cw - 1);
          T* dst = reinterpret_cast<T*>(buf + (w >> 1) * rs + pad8(j1));
          dst[w & 1] = val[u];
        }
      }
    }
  } else {
    for (int idx = threadIdx.x; idx < P1 * cw; idx += kThreads) {
      int j1 = idx >> lcw, c = idx & (cw - 1);
      int64_t j = (int64_t)P2 * j1 + j2_0 + c;
      cx<T> val{T(0), T(0)};
      if (MODE == kBlue) {
        if (j <= m) {
          T wgt = (j == 0 || j == m) ? T(1) : T(2);
          cx<T> ch = expmi<T>((j * j) % (2 * N), N);
          val = cscale(ch, wgt * (T)x[j]);
        }
      } else {  // kBSpec: conj(chirp) at lags -m..m, placed mod P
        int64_t t = j <= m ? j : (j >= P - m ? P - j : -1);
        if (t >= 0) val = cconj(expmi<T>((t * t) % (2 * N), N));
      }
      buf[c * rs + pad8(j1)] = val;
    }
  }
  __syncthreads();
  lds_fft<T, false>(buf, tw, l1, cw, rs);
  cx<T>* trow = tbuf + sg.t_off + (int64_t)row * sg.t_stride;
  const T invP = T(1) / (T)P;
  for (int idx = threadIdx.x; idx < P1 * cw; idx += kThreads) {
    int k1 = idx >> lcw, c = idx & (cw - 1);
    int64_t j2 = j2_0 + c;
    int64_t a = (j2 * k1) % P;
    cx<T> v = cmul(buf[c * rs + pad8(k1)], twiddle_P<T>(a, invP));
    trow[(int64_t)k1 * P2 + j2] = v;
  }
}

// ---- K2: row FFTs + spectral work + inverse row FFTs ----------------------
// One workgroup takes r2 consecutive k1 values of one row (TOD detector
// mode).  Real modes also load each partner row P1-k1, where the real-FFT
// unpacking partner C_(P-k) lives, so every element's partner is in LDS and
// one thread handles the pair (k, P-k) end to end: unpack, weight, repack,
// in place (w_L^(P-k) = -conj(w_L^k), so one sincospi per pair).
// TS: storage type of real spectra (the FP32 filter keeps FP32 spectra that
// were computed in FP64).
template <typename T, typename TS, int MODE>
__global__ void __launch_bounds__(kThreads, sizeof(T) == 4 ? 4 : 1) k2_kernel(const Seg* __restrict__ segs, int nseg,
                                                      cx<T>* __restrict__ tbuf) {
  extern __shared__ unsigned char smem_raw[];
  __shared__ int slot_k1[16], slot_partner[16];
  __shared__ int nslot_sh;
  const int s = find_seg(segs, nseg, blockIdx.x, 2);
  const Seg sg = segs[s];
  const int64_t local = (int64_t)blockIdx.x - sg.base2;
  const int row = (int)(local / sg.per2), grp = (int)(local % sg.per2);
  const int l2 = sg.l2, P1 = sg.p1, P2 = 1 << l2;
  const int rs = row_stride(P2);
  const int64_t P = (int64_t)P1 * P2;
  const bool real_mode = (MODE == kFilter || MODE == kFSpec);
  if (threadIdx.x == 0) {
    int ns = 0;
    const int kmax = real_mode ? P1 / 2 : P1 - 1;
    for (int q = 0; q < sg.r2; q++) {
      int k1 = grp * sg.r2 + q;
      if (k1 > kmax) break;
      int a = ns++;
      slot_k1[a] = k1;
      slot_partner[a] = a;
      int k1b = k1 == 0 ? 0 : P1 - k1;
      if (real_mode && k1b != k1) {
        int b = ns++;
        slot_k1[b] = k1b;
        slot_partner[a] = b;
        slot_partner[b] = a;
      }
    }
    nslot_sh = ns;
  }
  cx<T>* X = reinterpret_cast<cx<T>*>(smem_raw);             // [nslot][rs]
  cx<T>* tw = X + (real_mode ? 2 * sg.r2 : sg.r2) * rs;      // [P2] stage table
  // filter: this workgroup's spectrum rows, fetched with the T rows so their
  // latency overlaps the forward FFT ([nslot][P2] + B_P)
  TS* S = reinterpret_cast<TS*>(tw + P2);
  fill_stage_table<T>(tw, l2);
  __syncthreads();
  const int nslot = nslot_sh;
  cx<T>* trow = tbuf + sg.t_off + (int64_t)row * sg.t_stride;
  {
    constexpr int UNR = 8;
    const int total = nslot * P2;
    const TS* sbase = reinterpret_cast<const TS*>(sg.s_ptr) + (int64_t)row * sg.s_stride;
    for (int base = threadIdx.x; base < total; base += kThreads * UNR) {
      cx<T> v[UNR];
      TS b[UNR];
#pragma unroll
      for (int u = 0; u < UNR; u++) {
        int idx = base + u * kThreads;
        if (idx < total) {
          int64_t off = (int64_t)slot_k1[idx >> l2] * P2 + (idx & (P2 - 1));
          v[u] = trow[off];
          if (MODE == kFilter) b[u] = sbase[off];
        }
      }
#pragma unroll
      for (int u = 0; u < UNR; u++) {
        int idx = base + u * kThreads;
        if (idx < total) {
          X[(idx >> l2) * rs + pad8(idx & (P2 - 1))] = v[u];
          if (MODE == kFilter) S[idx] = b[u];
        }
      }
    }
    if (MODE == kFilter && threadIdx.x == 0) S[total] = sbase[P];
  }
  __syncthreads();
  lds_fft<T, false>(X, tw, l2, nslot, rs);
  auto at = [&](int idx) -> cx<T>& { return X[(idx >> l2) * rs + pad8(idx & (P2 - 1))]; };
  if (MODE == kBSpec) {
    cx<T>* srow = reinterpret_cast<cx<T>*>(sg.s_ptr);
    for (int idx = threadIdx.x; idx < nslot * P2; idx += kThreads)
      srow[(int64_t)slot_k1[idx >> l2] * P2 + (idx & (P2 - 1))] = at(idx);
    return;
  }
  if (MODE == kBlue) {
    const cx<T>* srow = reinterpret_cast<const cx<T>*>(sg.s_ptr);
    for (int idx = threadIdx.x; idx < nslot * P2; idx += kThreads)
      at(idx) = cmul(at(idx), srow[(int64_t)slot_k1[idx >> l2] * P2 + (idx & (P2 - 1))]);
    __syncthreads();
  } else {
    TS* srow = reinterpret_cast<TS*>(sg.s_ptr) + (int64_t)row * sg.s_stride;
    const T invP = T(1) / (T)P;
    for (int idx = threadIdx.x; idx < nslot * P2; idx += kThreads) {
      int sl = idx >> l2, k2 = idx & (P2 - 1);
      int kk1 = slot_k1[sl];
      int pidx = (kk1 == 0) ? (sl * P2 + ((P2 - k2) & (P2 - 1))) : (slot_partner[sl] * P2 + (P2 - 1 - k2));
      if (pidx < idx) continue;  // the pair is handled by its lower index
      int64_t k = kk1 + (int64_t)P1 * k2;
      cx<T> C = at(idx), Cq = at(pidx);
      // E_k = (C_k + conj C_(P-k))/2, O_k = (C_k - conj C_(P-k))/(2i); the
      // partner's E, O are conj(E_k), conj(O_k).
      cx<T> E = cscale(cadd(C, cconj(Cq)), T(0.5));
      cx<T> Dd = csub(C, cconj(Cq));
      cx<T> O = {Dd.im * T(0.5), -Dd.re * T(0.5)};
      cx<T> w = expmi2<T>(k, invP);  // w_L^k; w_L^(P-k) = -conj(w)
      cx<T> A = cadd(E, cmul(w, O));
      cx<T> Aq = csub(cconj(E), cmul(cconj(w), cconj(O)));
      int pk1 = slot_k1[pidx >> l2], pk2 = pidx & (P2 - 1);
      if (MODE == kFSpec) {
        srow[(int64_t)kk1 * P2 + k2] = (TS)A.re;
        if (pidx != idx) srow[(int64_t)pk1 * P2 + pk2] = (TS)Aq.re;  // self pair k = 0: Aq is A_P
        if (k == 0) srow[P] = (TS)(E.re - O.re);                       // A_P
        continue;
      }
      T b = (T)S[idx];
      T bq = (T)S[pidx];
      cx<T> Y = cscale(A, b), Yq = cscale(Aq, bq);
      if (k == 0) {
        // self pair: the inverse partner of Y_0 is Y_P (real)
        T yP = (E.re - O.re) * (T)S[nslot * P2];
        cx<T> Ep = {T(0.5) * (Y.re + yP), T(0.5) * Y.im};
        cx<T> Op = {T(0.5) * (Y.re - yP), T(0.5) * Y.im};
        at(idx) = {Ep.re - Op.im, Ep.im + Op.re};
        continue;
      }
      // D_k = E'_k + i O'_k, E'_k = (Y_k + conj Y_(P-k))/2,
      // O'_k = (Y_k - conj Y_(P-k)) conj(w_L^k)/2; same for P-k with w -> -conj(w)
      cx<T> Ep = cscale(cadd(Y, cconj(Yq)), T(0.5));
      cx<T> Op = cmul(cscale(csub(Y, cconj(Yq)), T(0.5)), cconj(w));
      cx<T> Eq = cscale(cadd(Yq, cconj(Y)), T(0.5));
      cx<T> Oq = cmul(cscale(csub(Yq, cconj(Y)), T(0.5)), cx<T>{-w.re, -w.im});
      at(idx) = {Ep.re - Op.im, Ep.im + Op.re};
      if (pidx != idx) at(pidx) = {Eq.re - Oq.im, Eq.im + Oq.re};
    }
    if (MODE == kFSpec) return;
    __syncthreads();
  }
  lds_fft<T, true>(X, tw, l2, nslot, rs);
  const T invP2 = T(1) / (T)P;
  for (int idx = threadIdx.x; idx < nslot * P2; idx += kThreads) {
    int sl = idx >> l2, j2 = idx & (P2 - 1);
    int kk1 = slot_k1[sl];
    int64_t a = ((int64_t)j2 * kk1) % P;
    trow[(int64_t)kk1 * P2 + j2] = cmul(at(idx), cconj(twiddle_P<T>(a, invP2)));
  }
}

// ---- Length classes of the 2^11-point-row engine ----------------------------
// A row of n samples belongs to the class P1, the smallest 5-smooth number in
// [2, 256] with 2^11 P1 >= 1.5 (n-1) + 1 (or a larger one of the caller's
// choice): the unit in which the autotuner compares and fixes transform
// lengths, and what mk_filt_plan_geometry reports.  The transform itself
// needs 2^11 q1 >= n only, two thirds of the class's length.
constexpr int kHotL2 = kRowL2;
constexpr int kHotP2 = kRowLen;
constexpr int ilog2c(int v) { return v <= 1 ? 0 : 1 + ilog2c(v >> 1); }
// Column tile of the general kernels: the largest power of two with
// cw P1 <= 4096.
constexpr int generic_cw(int p1) {
  int c = 1;
  while (2 * c * p1 <= kMaxWG && 2 * c <= kHotP2) c *= 2;
  return c;
}
constexpr int kHotP1[] = {2,   3,   4,   5,   6,   8,   9,   10,  12,  15,  16,  18,  20,  24,  25,  27,  30,
                          32,  36,  40,  45,  48,  50,  54,  60,  64,  72,  75,  80,  81,  90,  96,  100, 108,
                          120, 125, 128, 135, 144, 150, 160, 162, 180, 192, 200, 216, 225, 240, 243, 250, 256};
constexpr int kNumHotP1 = sizeof(kHotP1) / sizeof(kHotP1[0]);
int hot_p1_index(int p1) {
  for (int i = 0; i < kNumHotP1; i++)
    if (kHotP1[i] == p1) return i;
  return -1;
}

// ---- K3: inverse column FFTs + output -------------------------------------
template <typename T, typename TOut, int MODE>
__global__ void __launch_bounds__(kThreads, sizeof(T) == 4 ? 4 : 1) k3_kernel(const Seg* __restrict__ segs, int nseg,
                                                      const cx<T>* __restrict__ tbuf, TOut* __restrict__ out) {
  extern __shared__ unsigned char smem_raw[];
  const int s = find_seg(segs, nseg, blockIdx.x, 3);
  const Seg sg = segs[s];
  const int64_t local = (int64_t)blockIdx.x - sg.base3;
  const int row = (int)(local / sg.per1), jb = (int)(local % sg.per1);
  // power-of-two column lengths only (the plan routes mixed lengths to the
  // hot path)
  const int l1 = sg.l1, l2 = sg.l2, P1 = 1 << l1, P2 = 1 << l2, cw = sg.cw;
  const int lcw = 31 - __clz(cw);
  const int rs = row_stride(P1);
  const int64_t P = (int64_t)P1 * P2;
  const int64_t m = sg.n - 1, N = 2 * m;
  cx<T>* buf = reinterpret_cast<cx<T>*>(smem_raw);  // [cw][rs]
  cx<T>* tw = buf + cw * rs;                          // [P1] stage table
  const cx<T>* trow = tbuf + sg.t_off + (int64_t)row * sg.t_stride;
  const int j2_0 = jb * cw;
  fill_stage_table<T>(tw, l1);
  {
    constexpr int UNR = 8;
    const int total = P1 * cw;
    for (int base = threadIdx.x; base < total; base += kThreads * UNR) {
      cx<T> v[UNR];
#pragma unroll
      for (int u = 0; u < UNR; u++) {
        int idx = base + u * kThreads;
        if (idx < total) {
          int k1 = idx >> lcw, c = idx & (cw - 1);
          v[u] = trow[(int64_t)k1 * P2 + j2_0 + c];
        }
      }
#pragma unroll
      for (int u = 0; u < UNR; u++) {
        int idx = base + u * kThreads;
        if (idx < total) {
          int k1 = idx >> lcw, c = idx & (cw - 1);
          buf[c * rs + pad8(k1)] = v[u];
        }
      }
    }
  }
  __syncthreads();
  lds_fft<T, true>(buf, tw, l1, cw, rs);
  const T scale = T(1) / (T)P;
  TOut* y = out + sg.out_off + (int64_t)row * sg.out_stride;
  if (MODE == kFilter) {
    const bool halve = sg.flags & 1;
    for (int idx = threadIdx.x; idx < P1 * cw * 2; idx += kThreads) {
      int j1 = idx >> (lcw + 1), w = idx & (2 * cw - 1);
      int64_t i = 2 * ((int64_t)P2 * j1 + j2_0) + w;
      int64_t k = i - m;
      if (k >= 0 && k <= m) {
        const T* src = reinterpret_cast<const T*>(buf + (w >> 1) * rs + pad8(j1));
        T v = src[w & 1] * scale;
        if (halve && (k == 0 || k == m)) v *= T(0.5);
        y[k] = (TOut)v;
      }
    }
  } else {  // kBlue
    for (int idx = threadIdx.x; idx < P1 * cw; idx += kThreads) {
      int j1 = idx >> lcw, c = idx & (cw - 1);
      int64_t k = (int64_t)P2 * j1 + j2_0 + c;
      if (k <= m) {
        cx<T> w = cscale(buf[c * rs + pad8(j1)], scale);
        cx<T> ch = expmi<T>((k * k) % (2 * N), N);
        y[k] = (TOut)(ch.re * w.re - ch.im * w.im);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Host-side planning

int log2_ceil(int64_t x) {
  int q = 0;
  while ((int64_t(1) << q) < x) q++;
  return q;
}

struct Geometry {
  int l1, l2, cw;  // l1 = log2(p1), or -1 when p1 is not a power of two
  int p1;
  int64_t P;
};

// P = 2^q complex points split as P1 * P2 with the row length P2 as long as
// K2 holds (2^11 points, a real-mode row and its partner fill one
// workgroup), so the columns are short and K1/K3 can take many adjacent
// columns at once: their global accesses are runs of cw complex points.
// MK_FFT_L2MAX (power-of-two exponent, 2..11) lowers the row-length cap.
//
// mixed: the FP32 hot path takes any 5-smooth P1 in [2, 256] with P2 = 2^11,
// so P = P1 2^11 is the smallest such multiple of 2^11 >= P_min (instead of
// the next power of two): about 1.4x fewer points on average.
Geometry hot_geometry(int p1) {
  Geometry g;
  g.p1 = p1;
  g.l1 = (p1 & (p1 - 1)) == 0 ? ilog2c(p1) : -1;
  g.l2 = kHotL2;
  g.P = (int64_t)p1 * kHotP2;
  g.cw = generic_cw(p1);
  return g;
}

Geometry geometry(int64_t P_min, int elem_bytes, bool mixed = false) {
  if (mixed && P_min > kHotP2) {  // a length class of the 2^11-point-row engine
    const int64_t need = (P_min + kHotP2 - 1) / kHotP2;
    for (int i = 0; i < kNumHotP1; i++)
      if (kHotP1[i] >= need) return hot_geometry(kHotP1[i]);
  }
  int q = std::max(2, log2_ceil(P_min));
  static int l2max = [] {
    const char* e = getenv("MK_FFT_L2MAX");
    int v = e ? atoi(e) : 11;
    return std::min(11, std::max(2, v));
  }();
  Geometry g;
  g.l2 = std::min(l2max, q - 1);
  g.l1 = q - g.l2;
  g.p1 = 1 << g.l1;
  g.P = int64_t(1) << q;
  int P1 = g.p1, P2 = 1 << g.l2;
  int cw = std::min(std::max(1, kMaxWG / P1), P2);
  // keep the K1/K3 tile plus the twiddle table within the LDS budget
  while (cw > 1 && ((int64_t)cw * row_stride(P1) + P1) * 2 * elem_bytes > kMaxLds) cw >>= 1;
  g.cw = cw;
  return g;
}

template <typename K>
void allow_big_lds(K kernel) {
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                            kMaxLds);
}

void allow_lds_all() {
  static bool done = false;
  if (done) return;
  done = true;
  allow_big_lds(k1_kernel<float, float, kFilter>);
  allow_big_lds(k1_kernel<double, double, kFilter>);
  allow_big_lds(k1_kernel<float, double, kFSpec>);
  allow_big_lds(k1_kernel<double, double, kFSpec>);
  allow_big_lds(k1_kernel<float, float, kBlue>);
  allow_big_lds(k1_kernel<double, double, kBlue>);
  allow_big_lds(k1_kernel<float, float, kBSpec>);
  allow_big_lds(k1_kernel<double, double, kBSpec>);
  allow_big_lds(k2_kernel<float, float, kFilter>);
  allow_big_lds(k2_kernel<double, double, kFilter>);
  allow_big_lds(k2_kernel<float, float, kFSpec>);
  allow_big_lds(k2_kernel<double, double, kFSpec>);
  allow_big_lds(k2_kernel<double, float, kFSpec>);
  allow_big_lds(k2_kernel<float, float, kBlue>);
  allow_big_lds(k2_kernel<double, double, kBlue>);
  allow_big_lds(k2_kernel<float, float, kBSpec>);
  allow_big_lds(k2_kernel<double, double, kBSpec>);
  allow_big_lds(k3_kernel<float, float, kFilter>);
  allow_big_lds(k3_kernel<double, double, kFilter>);
  allow_big_lds(k3_kernel<float, float, kBlue>);
  allow_big_lds(k3_kernel<double, double, kBlue>);
  allow_rows_lds();
  (void)hipGetLastError();  // an unsupported attribute must not poison later launch checks
}

size_t lds_k13(const Geometry& g, int eb) {
  return (size_t)(g.cw * row_stride(g.p1) + g.p1) * 2 * eb;
}
// k1 values per K2 workgroup: slots (2 per k1 for real modes) * P2 <= kMaxWG
// LDS of K2: slot rows, the stage table and (real modes) the slots' spectrum
// values, one real each plus B_P.
size_t k2_bytes(int r, int P2, int eb, bool real) {
  int ns = real ? 2 * r : r;
  return (size_t)(ns * row_stride(P2) + P2) * 2 * eb + (real ? (size_t)(ns * P2 + 1) * eb : 0) + 64;
}
// k1 values per K2 workgroup: slots (2 per k1 for real modes) * P2 <= kMaxWG
int k2_r2(const Geometry& g, int eb, bool real) {
  int P2 = 1 << g.l2, P1 = g.p1;
  int r = 8;
  while (r > 1 && ((real ? 2 : 1) * r * P2 > kMaxWG || k2_bytes(r, P2, eb, real) > (size_t)kMaxLds)) r >>= 1;
  return std::min(r, real ? P1 / 2 + 1 : P1);
}
size_t lds_k2(const Geometry& g, int eb, bool real = true) {
  return k2_bytes(k2_r2(g, eb, real), 1 << g.l2, eb, real);
}

}  // namespace

// ---------------------------------------------------------------------------
// Filter plan: per segment (TOD) rows x n, input/output row offsets.

struct mk_filt_plan {
  int nseg = 0;
  int elem_bytes = 4;  // 4: FP32 spectra and T buffer, 8: FP64
  std::vector<Seg> h_segs;
  int64_t n1 = 0, n2 = 0;  // total K1/K3 items, K2 items
  int64_t t_elems = 0, s_elems = 0;  // complex values of the work buffer, reals of the spectra
  void* tbuf = nullptr;    // complex
  bool tbuf_owned = true;  // false: the caller's buffer (mk_filt_plan_set_work)
  void* spec = nullptr;    // real: 2 (P+2) per row on the 2^11-row path, P+1 on the general one
  size_t lds1 = 0, lds2 = 0;  // LDS of the general kernels
  bool have_spec = false;
  std::vector<char> borrowed;
  // Segments on the 2^11-row path (one list for the row pass and one grouped
  // by column count for the column passes, a launch per count) and the rest,
  // each list with its own work-item numbering.
  Seg* d_hot = nullptr;
  Seg* d_hotc = nullptr;
  Seg* d_cold = nullptr;
  int nhot = 0, ncold = 0;
  int64_t n2hot = 0, n2cold = 0, n1cold = 0;
  int g_off[kNumQ1] = {0}, g_cnt[kNumQ1] = {0};  // per column count (kQ1 index)
  int64_t g_n1[kNumQ1] = {0};
  // twiddle tables in the plan's precision, and in FP64 for the spectrum pass
  // of an FP32 plan (freed after it): the common ones, then one per count
  void* tw = nullptr;
  int64_t g_tab[kNumQ1] = {0};  // element offset of a count's table
  int64_t tw_elems = 0, tw_all = 0;  // complex elements without / with the end-mode phases
};

namespace {
// The work buffer (rows * P complex) is allocated on first use and can be
// released between uses; spectra stay resident.
int ensure_tbuf(const mk_filt_plan* cp) {
  mk_filt_plan* p = const_cast<mk_filt_plan*>(cp);
  if (p->tbuf) return MK_OK;
  p->tbuf_owned = true;
  if (hipMalloc(&p->tbuf, std::max<int64_t>(1, p->t_elems) * 2 * p->elem_bytes) != hipSuccess) {
    p->tbuf = nullptr;
    mk::set_error("filter plan: work buffer allocation (%lld B) failed", (long long)(p->t_elems * 2 * p->elem_bytes));
    return MK_ERR_ALLOC;
  }
  return MK_OK;
}

// Uploads the segment lists; eb: precision of the passes they number (the
// column tile depends on it).
int upload_lists(mk_filt_plan* p, int eb) {
  std::vector<Seg> hot, cold, hotc;
  int64_t b_hot = 0, b_cold2 = 0, b_cold1 = 0;
  for (const Seg& s0 : p->h_segs) {
    Seg s = s0;
    if (s.hot) {
      s.tw_off = p->g_tab[q1_index(s.q1)];
      s.per2 = (s.q1 + 1) / 2;  // pairs (k1, q1-k1), k1 = 1..; column 0 (+ q1/2) in item 0
      s.base2 = b_hot;
      b_hot += (int64_t)s.rows * s.per2;
      hot.push_back(s);
    } else {
      s.base2 = b_cold2;
      b_cold2 += (int64_t)s.rows * s.per2;
      s.base1 = s.base3 = b_cold1;
      b_cold1 += (int64_t)s.rows * s.per1;
      cold.push_back(s);
    }
  }
  for (int l = 0; l < kNumQ1; l++) {
    p->g_off[l] = (int)hotc.size();
    int64_t b = 0;
    for (const Seg& s0 : hot)
      if (s0.q1 == kQ1[l]) {
        Seg s = s0;
        s.base1 = s.base3 = b;
        b += (int64_t)s.rows * (eb == 4 ? col_blocks<float>(s.q1) : col_blocks<double>(s.q1));
        hotc.push_back(s);
      }
    p->g_cnt[l] = (int)hotc.size() - p->g_off[l];
    p->g_n1[l] = b;
  }
  p->nhot = (int)hot.size();
  p->ncold = (int)cold.size();
  p->n2hot = b_hot;
  p->n2cold = b_cold2;
  p->n1cold = b_cold1;
  if ((p->nhot && hipMemcpy(p->d_hot, hot.data(), hot.size() * sizeof(Seg), hipMemcpyHostToDevice) != hipSuccess) ||
      (p->nhot && hipMemcpy(p->d_hotc, hotc.data(), hotc.size() * sizeof(Seg), hipMemcpyHostToDevice) != hipSuccess) ||
      (p->ncold && hipMemcpy(p->d_cold, cold.data(), cold.size() * sizeof(Seg), hipMemcpyHostToDevice) != hipSuccess)) {
    mk::set_error("filter plan: descriptor upload failed");
    return MK_ERR_HIP;
  }
  return MK_OK;
}
int upload(mk_filt_plan* p) { return upload_lists(p, p->elem_bytes); }

// The tables a plan uses: the common ones, then one per column count, then
// the end-mode phases per row length (of one column count).
void layout_tables(mk_filt_plan* p) {
  p->tw_elems = 0;
  for (Seg& s : p->h_segs) {
    if (!s.hot) continue;
    if (p->tw_elems == 0) p->tw_elems = kTwCommon;
    const int i = q1_index(s.q1);
    if (!p->g_tab[i]) {
      p->g_tab[i] = p->tw_elems;
      p->tw_elems += q1_table_elems(s.q1);
    }
  }
  p->tw_all = p->tw_elems;
  for (size_t i = 0; i < p->h_segs.size(); i++) {
    Seg& s = p->h_segs[i];
    if (!s.hot) continue;
    s.em_off = 0;
    for (size_t k = 0; k < i && !s.em_off; k++) {
      const Seg& o = p->h_segs[k];
      if (o.hot && o.n == s.n && o.q1 == s.q1) s.em_off = o.em_off;
    }
    if (!s.em_off) {
      s.em_off = p->tw_all;
      p->tw_all += end_phase_elems(s.q1);
    }
  }
}

// Builds the twiddle tables in precision T into tab (tw_elems values).
template <typename T>
int build_tables(const mk_filt_plan* p, void* tab, hipStream_t st) {
  bool first = true;
  for (int i = 0; i < kNumQ1; i++)
    if (p->g_tab[i]) {
      launch_col_tables<T>(kQ1[i], first ? (cx<T>*)tab : nullptr, (cx<T>*)tab + p->g_tab[i], st);
      first = false;
    }
  return mk::check_launch("col_tables_kernel");
}
template <typename T>
int build_end_phases(const mk_filt_plan* p, hipStream_t st) {
  int64_t next = p->tw_elems;
  for (const Seg& s : p->h_segs)
    if (s.hot && s.em_off == next) {  // a length's first segment
      launch_end_phases<T>((cx<T>*)p->tw + next, s.n, s.q1, st);
      next += end_phase_elems(s.q1);
    }
  return mk::check_launch("end_phase_kernel");
}

void free_filt(mk_filt_plan* p) {
  if (!p) return;
  if (p->d_hot) (void)hipFree(p->d_hot);
  if (p->d_hotc) (void)hipFree(p->d_hotc);
  if (p->d_cold) (void)hipFree(p->d_cold);
  if (p->tw) (void)hipFree(p->tw);
  if (p->tbuf && p->tbuf_owned) (void)hipFree(p->tbuf);
  if (p->spec) (void)hipFree(p->spec);
  delete p;
}

// desc per segment: {rows, n, in_off, in_stride, out_off, out_stride}
// mixed: FP32 filter plans, whose geometry is reported in length classes.
// hot: rows longer than 2^11 * 2/3 samples and up to 2^19 take the
// 2^11-point-row engine.
// p1 (may be null): per segment a hot column length chosen by the caller
// (0 = the default, the smallest one that fits).
int build_segs(int nseg, const int64_t* desc, int eb, bool filter, std::vector<Seg>& segs, int64_t* n1,
               int64_t* n2, int64_t* t_elems, int64_t* s_elems, size_t* lds1, size_t* lds2, bool mixed = false,
               const int32_t* p1 = nullptr, bool hot = false) {
  segs.clear();
  int64_t b1 = 0, b2 = 0, toff = 0, soff = 0;
  size_t l1max = 0, l2max = 0;
  for (int i = 0; i < nseg; i++) {
    const int64_t* d = desc + 6 * i;
    int64_t rows = d[0], n = d[1];
    MK_REQUIRE(rows >= 0 && n >= 2 && n < (int64_t(1) << 30), MK_ERR_ARG,
               "segment %d: need rows >= 0 and 2 <= n < 2^30 (rows=%lld n=%lld)", i, (long long)rows,
               (long long)n);
    int64_t m = n - 1;
    const int64_t P_min = filter ? (3 * m + 2) / 2 : 2 * m + 1;
    Geometry g = geometry(P_min, eb, mixed);
    const int p1_min = g.p1;
    if (p1 && p1[i] > 0) {
      MK_REQUIRE(mixed && hot_p1_index(p1[i]) >= 0, MK_ERR_ARG,
                 "segment %d: column length %d is not one of the FP32 hot lengths", i, (int)p1[i]);
      MK_REQUIRE((int64_t)p1[i] * kHotP2 >= P_min && P_min > kHotP2, MK_ERR_ARG,
                 "segment %d: column length %d is too short for n=%lld", i, (int)p1[i], (long long)n);
      g = hot_geometry(p1[i]);
    }
    MK_REQUIRE(g.P <= (int64_t(1) << 24), MK_ERR_ARG, "segment %d: n=%lld too long", i, (long long)n);
    Seg s{};
    s.in_off = d[2]; s.in_stride = d[3]; s.out_off = d[4]; s.out_stride = d[5];
    s.rows = (int32_t)rows; s.n = (int32_t)n; s.l1 = g.l1; s.l2 = g.l2; s.cw = g.cw; s.flags = 0; s.p1 = g.p1;
    // the engine's own length: 2^11 q1 >= n, and for a longer class than the
    // default two thirds of its columns
    s.q1 = 0;
    if (hot && filter && P_min > kHotP2) {
      const int64_t cls = p1 && p1[i] > p1_min ? mk::cdiv(2 * (int64_t)p1[i], 3) * kHotP2 : 0;
      s.q1 = q1_at_least(std::max(m + 1, cls));
    }
    s.hot = s.q1 > 0;
    const int64_t P = s.hot ? (int64_t)s.q1 * kHotP2 : g.P;
    const int64_t s_row = s.hot ? 2 * (P + 2) : P + 1;
    s.t_off = toff; s.t_stride = P;
    s.s_off = soff; s.s_stride = filter ? s_row : 0;
    s.per1 = (int32_t)((int64_t(1) << g.l2) / g.cw);
    s.r2 = k2_r2(g, 8, filter);  // same grouping for FP32 and FP64 passes
    s.per2 = (int32_t)mk::cdiv(filter ? g.p1 / 2 + 1 : g.p1, s.r2);
    s.base1 = b1; s.base2 = b2; s.base3 = b1;
    b1 += rows * s.per1;
    b2 += rows * s.per2;
    toff += rows * P;
    soff += filter ? rows * s_row : P;
    if (!s.hot) {
      l1max = std::max(l1max, lds_k13(g, eb));
      l2max = std::max(l2max, lds_k2(g, eb, filter));
    }
    MK_REQUIRE(l1max <= (size_t)kMaxLds && l2max <= (size_t)kMaxLds, MK_ERR_ARG,
               "segment %d: n=%lld needs more LDS than the %d-byte budget at %d-byte precision", i,
               (long long)n, kMaxLds, eb);
    segs.push_back(s);
  }
  for (Seg& s : segs) {  // behind the rows: one value per row of the 2^11-row path
    s.e_off = toff;
    if (s.hot) toff += s.rows;
  }
  *n1 = b1; *n2 = b2; *t_elems = toff; *s_elems = soff; *lds1 = l1max; *lds2 = l2max;
  return MK_OK;
}

// Spectrum pass of the general path in arithmetic type T into spectra of type
// TS; lds1/lds2 sized for T.
template <typename T, typename TS>
void launch_fspec(mk_filt_plan* p, const void* wdct, void* tb, size_t lds1, size_t lds2, hipStream_t st) {
  k1_kernel<T, double, kFSpec><<<(unsigned)p->n1cold, kThreads, lds1, st>>>(p->d_cold, p->ncold, (const double*)wdct,
                                                                            (cx<T>*)tb);
  k2_kernel<T, TS, kFSpec><<<(unsigned)p->n2cold, kThreads, lds2, st>>>(p->d_cold, p->ncold, (cx<T>*)tb);
}

// The 2^11-row path's column passes over every column count of the plan.
template <typename T>
void launch_hot_fwd(const mk_filt_plan* p, int mode, const void* in, cx<T>* tb, const cx<T>* tw, int comp,
                    hipStream_t st) {
  for (int i = 0; i < kNumQ1; i++)
    if (p->g_n1[i])
      launch_cols_fwd<T>(kQ1[i], mode, p->d_hotc + p->g_off[i], p->g_cnt[i], p->g_n1[i], in, tb,
                         tw, tw + p->g_tab[i] + kQ1[i] * kRowTw, nullptr, comp, st);
}

template <typename T, typename TIO>
void launch_filter(const mk_filt_plan* p, const TIO* in, TIO* out, hipStream_t st) {
  cx<T>* tb = (cx<T>*)p->tbuf;
  const cx<T>* tw = (const cx<T>*)p->tw;
  launch_hot_fwd<T>(p, kFilter, in, tb, tw, 0, st);
  if (p->n1cold)
    k1_kernel<T, TIO, kFilter><<<(unsigned)p->n1cold, kThreads, p->lds1, st>>>(p->d_cold, p->ncold, in, tb);
  if (p->n2hot) launch_rows<T>(kFilter, p->d_hot, p->nhot, p->n2hot, tb, tw, 0, false, st);
  if (p->n2cold)
    k2_kernel<T, T, kFilter><<<(unsigned)p->n2cold, kThreads, p->lds2, st>>>(p->d_cold, p->ncold, tb);
  for (int i = 0; i < kNumQ1; i++)
    if (p->g_n1[i])
      launch_cols_inv<T>(kQ1[i], kFilter, p->d_hotc + p->g_off[i], p->g_cnt[i], p->g_n1[i], tb, out,
                         tw, tw + p->g_tab[i] + kQ1[i] * kRowTw, nullptr, st);
  if (p->n1cold)
    k3_kernel<T, TIO, kFilter><<<(unsigned)p->n1cold, kThreads, p->lds1, st>>>(p->d_cold, p->ncold, tb, out);
}

}  // namespace

extern "C" int mk_filt_plan_create(int nseg, const int64_t* desc, int elem_bytes, mk_filt_plan** out) {
  return mk_filt_plan_create_p1(nseg, desc, elem_bytes, nullptr, out);
}

extern "C" int mk_filt_hot_p1(int32_t* out, int cap) {
  if (out)
    for (int i = 0; i < kNumHotP1 && i < cap; i++) out[i] = kHotP1[i];
  return kNumHotP1;
}

extern "C" int mk_filt_plan_create_p1(int nseg, const int64_t* desc, int elem_bytes, const int32_t* p1,
                                      mk_filt_plan** out) {
  MK_REQUIRE(out, MK_ERR_ARG, "out is NULL");
  *out = nullptr;
  MK_REQUIRE(nseg >= 0 && (nseg == 0 || desc), MK_ERR_ARG, "bad segment table");
  MK_REQUIRE(elem_bytes == 4 || elem_bytes == 8, MK_ERR_ARG, "elem_bytes must be 4 or 8");
  allow_lds_all();
  mk_filt_plan* p = new mk_filt_plan();
  p->nseg = nseg;
  p->borrowed.assign(std::max(1, nseg), 0);
  p->elem_bytes = elem_bytes;
  const bool hot = getenv("MK_FFT_NO_HOT") == nullptr;
  int st = build_segs(nseg, desc, elem_bytes, true, p->h_segs, &p->n1, &p->n2, &p->t_elems, &p->s_elems, &p->lds1,
                      &p->lds2, hot && elem_bytes == 4, p1, hot);
  if (st) { free_filt(p); return st; }
  MK_REQUIRE(p->n1 < INT32_MAX && p->n2 < INT32_MAX, (free_filt(p), MK_ERR_ARG), "too many work items");
  layout_tables(p);
  if (hipMalloc((void**)&p->d_hot, std::max<size_t>(1, nseg) * sizeof(Seg)) != hipSuccess ||
      hipMalloc((void**)&p->d_hotc, std::max<size_t>(1, nseg) * sizeof(Seg)) != hipSuccess ||
      hipMalloc((void**)&p->d_cold, std::max<size_t>(1, nseg) * sizeof(Seg)) != hipSuccess ||
      hipMalloc(&p->tw, std::max<int64_t>(1, p->tw_all) * 2 * elem_bytes) != hipSuccess) {
    free_filt(p);
    mk::set_error("filter plan: device allocation failed");
    return MK_ERR_ALLOC;
  }
  // spectra are allocated by mk_filt_plan_set_weights: a plan that borrows
  // every segment's spectrum never holds any of its own
  for (auto& sg : p->h_segs) sg.s_ptr = nullptr;
  if (p->tw_elems) {
    st = elem_bytes == 4 ? build_tables<float>(p, p->tw, nullptr) : build_tables<double>(p, p->tw, nullptr);
    if (st == MK_OK) st = elem_bytes == 4 ? build_end_phases<float>(p, nullptr) : build_end_phases<double>(p, nullptr);
    if (st == MK_OK && hipDeviceSynchronize() != hipSuccess)  // exec may run on another stream
      st = (mk::set_error("filter plan: twiddle table build failed"), MK_ERR_HIP);
    if (st) { free_filt(p); return st; }
  }
  if (upload(p)) {
    free_filt(p);
    return MK_ERR_HIP;
  }
  *out = p;
  return MK_OK;
}

extern "C" int mk_filt_plan_borrow_spectrum(mk_filt_plan* p, int seg, const mk_filt_plan* src, int src_seg) {
  MK_REQUIRE(p && src, MK_ERR_ARG, "null plan");
  MK_REQUIRE(seg >= 0 && seg < p->nseg && src_seg >= 0 && src_seg < src->nseg, MK_ERR_ARG, "segment out of range");
  MK_REQUIRE(p->elem_bytes == src->elem_bytes, MK_ERR_ARG, "precision mismatch");
  MK_REQUIRE(src->have_spec, MK_ERR_ARG, "source plan has no weights");
  Seg& d = p->h_segs[seg];
  const Seg& s = src->h_segs[src_seg];
  MK_REQUIRE(d.rows == s.rows && d.n == s.n && d.p1 == s.p1 && d.l2 == s.l2 && d.q1 == s.q1, MK_ERR_ARG,
             "segment geometry differs (rows %d/%d, n %d/%d)", d.rows, s.rows, d.n, s.n);
  d.s_ptr = s.s_ptr;
  p->borrowed[seg] = 1;
  bool all = true;
  for (int i = 0; i < p->nseg; i++) all = all && p->borrowed[i];
  if (all) p->have_spec = true;
  return upload(p) ? MK_ERR_HIP : MK_OK;
}

extern "C" int mk_filt_plan_destroy(mk_filt_plan* p) {
  free_filt(p);
  return MK_OK;
}

extern "C" int mk_filt_plan_info(const mk_filt_plan* p, int64_t* info) {
  MK_REQUIRE(p && info, MK_ERR_ARG, "null pointer");
  info[0] = p->nseg;
  info[1] = p->n1;
  info[2] = p->n2;
  info[3] = p->t_elems * 2 * p->elem_bytes;
  info[4] = p->s_elems * p->elem_bytes;
  info[5] = p->elem_bytes;
  info[6] = (int64_t)p->lds1;
  info[7] = (int64_t)p->lds2;
  return MK_OK;
}

// Per-segment geometry: out[4*i..] = {P1, P2, cw, P1 P2} of segment i (on the
// 2^11-row path the length class, see kHotP1).
extern "C" int mk_filt_plan_geometry(const mk_filt_plan* p, int64_t* out) {
  MK_REQUIRE(p && out, MK_ERR_ARG, "null pointer");
  for (int i = 0; i < p->nseg; i++) {
    const Seg& s = p->h_segs[i];
    out[4 * i] = s.p1;
    out[4 * i + 1] = int64_t(1) << s.l2;
    out[4 * i + 2] = s.cw;
    out[4 * i + 3] = (int64_t)s.p1 << s.l2;
  }
  return MK_OK;
}

extern "C" int mk_filt_plan_set_weights(mk_filt_plan* p, const double* wdct, void* stream) {
  MK_REQUIRE(p && (p->nseg == 0 || wdct), MK_ERR_ARG, "null argument");
  for (int i = 0; i < p->nseg; i++)
    MK_REQUIRE(!p->borrowed[i], MK_ERR_ARG, "plan borrows spectra; set_weights would overwrite the source plan");
  if (p->n1 == 0) { p->have_spec = true; return MK_OK; }
  hipStream_t st = mk::as_stream(stream);
  if (!p->spec) {
    if (hipMalloc(&p->spec, std::max<int64_t>(1, p->s_elems) * p->elem_bytes) != hipSuccess) {
      p->spec = nullptr;
      mk::set_error("filter plan: spectrum allocation (%lld B) failed", (long long)(p->s_elems * p->elem_bytes));
      return MK_ERR_ALLOC;
    }
    for (auto& sg : p->h_segs) sg.s_ptr = (unsigned char*)p->spec + sg.s_off * p->elem_bytes;
    int r = upload(p);
    if (r) return r;
  }
  // The spectrum is always computed in FP64 (a transient FP64 work buffer)
  // and stored in the plan's precision, unless FP64 LDS tiles of the general
  // path would not fit.
  size_t l1_64 = 0, l2_64 = 0;
  for (const Seg& sg : p->h_segs) {
    if (sg.hot) continue;
    Geometry g{sg.l1, sg.l2, sg.cw, sg.p1, (int64_t)sg.p1 << sg.l2};
    l1_64 = std::max(l1_64, lds_k13(g, 8));
    l2_64 = std::max(l2_64, lds_k2(g, 8));
  }
  const bool fp64_pass = l1_64 <= (size_t)kMaxLds && l2_64 <= (size_t)kMaxLds;
  void* tb = nullptr;
  void* tw64 = nullptr;
  int r = MK_OK;
  if (hipMalloc(&tb, std::max<int64_t>(1, p->t_elems) * 16) != hipSuccess ||
      (p->elem_bytes == 4 && p->tw_elems && hipMalloc(&tw64, p->tw_elems * 16) != hipSuccess)) {
    if (tb) (void)hipFree(tb);
    mk::set_error("filter plan: spectrum work allocation (%lld B) failed", (long long)(p->t_elems * 16));
    return MK_ERR_ALLOC;
  }
  if (p->n2hot) {
    if (p->elem_bytes == 4) {  // the FP64 pass numbers its column tiles differently
      r = build_tables<double>(p, tw64, st);
      if (r == MK_OK) r = upload_lists(p, 8);
    }
    const cx<double>* tw = (const cx<double>*)(p->elem_bytes == 4 ? tw64 : p->tw);
    for (int comp = 0; comp < 2 && r == MK_OK; comp++) {
      launch_hot_fwd<double>(p, kFSpec, wdct, (cx<double>*)tb, tw, comp, st);
      launch_rows<double>(kFSpec, p->d_hot, p->nhot, p->n2hot, (cx<double>*)tb, tw, comp, p->elem_bytes == 4, st);
      r = mk::check_launch("filter spectrum");
    }
    int64_t rows = 0;
    for (const Seg& sg : p->h_segs) rows += sg.hot ? sg.rows : 0;
    if (r == MK_OK) {
      launch_end_modes(p->d_hot, p->nhot, rows, wdct, p->elem_bytes == 4, st);
      r = mk::check_launch("end_modes_kernel");
    }
  }
  if (p->n1cold && r == MK_OK) {
    if (fp64_pass && p->elem_bytes == 4) launch_fspec<double, float>(p, wdct, tb, l1_64, l2_64, st);
    else if (fp64_pass) launch_fspec<double, double>(p, wdct, tb, l1_64, l2_64, st);
    else launch_fspec<float, float>(p, wdct, tb, p->lds1, p->lds2, st);
    r = mk::check_launch("filter spectrum");
  }
  if (hipStreamSynchronize(st) != hipSuccess && r == MK_OK)
    r = (mk::set_error("filter spectrum: stream synchronisation failed"), MK_ERR_HIP);
  if (p->n2hot && p->elem_bytes == 4) {  // back to the FP32 numbering
    const int u = upload(p);
    if (r == MK_OK) r = u;
  }
  (void)hipFree(tb);
  if (tw64) (void)hipFree(tw64);
  if (r == MK_OK) p->have_spec = true;
  return r;
}

extern "C" int mk_filt_plan_exec_f32(const mk_filt_plan* p, const float* in, float* out, void* stream) {
  MK_REQUIRE(p && in && out, MK_ERR_ARG, "null argument");
  MK_REQUIRE(p->have_spec, MK_ERR_ARG, "filter weights not set");
  MK_REQUIRE(p->elem_bytes == 4, MK_ERR_ARG, "plan was created for FP64");
  if (p->n1 == 0) return MK_OK;
  int r = ensure_tbuf(p);
  if (r) return r;
  launch_filter<float, float>(p, in, out, mk::as_stream(stream));
  return mk::check_launch("filter exec f32");
}

extern "C" int mk_filt_plan_exec_f64(const mk_filt_plan* p, const double* in, double* out, void* stream) {
  MK_REQUIRE(p && in && out, MK_ERR_ARG, "null argument");
  MK_REQUIRE(p->have_spec, MK_ERR_ARG, "filter weights not set");
  MK_REQUIRE(p->elem_bytes == 8, MK_ERR_ARG, "plan was created for FP32");
  if (p->n1 == 0) return MK_OK;
  int r = ensure_tbuf(p);
  if (r) return r;
  launch_filter<double, double>(p, in, out, mk::as_stream(stream));
  return mk::check_launch("filter exec f64");
}

extern "C" int mk_filt_plan_release_work(mk_filt_plan* p, void* stream) {
  MK_REQUIRE(p, MK_ERR_ARG, "null plan");
  if (p->tbuf) {
    MK_HIP(hipStreamSynchronize(mk::as_stream(stream)));
    if (p->tbuf_owned) MK_HIP(hipFree(p->tbuf));
    p->tbuf = nullptr;
  }
  return MK_OK;
}

extern "C" int mk_filt_plan_work_bytes(const mk_filt_plan* p, int64_t* bytes) {
  MK_REQUIRE(p && bytes, MK_ERR_ARG, "null pointer");
  *bytes = p->t_elems * 2 * p->elem_bytes;
  return MK_OK;
}

extern "C" int mk_filt_plan_set_work(mk_filt_plan* p, void* work, int64_t bytes, void* stream) {
  MK_REQUIRE(p, MK_ERR_ARG, "null plan");
  const int64_t need = p->t_elems * 2 * p->elem_bytes;
  MK_REQUIRE(work == nullptr || (bytes >= need && ((uintptr_t)work & 15) == 0), MK_ERR_ARG,
             "work buffer of %lld B (need %lld B, 16-byte aligned)", (long long)bytes, (long long)need);
  int r = mk_filt_plan_release_work(p, stream);
  if (r) return r;
  if (work) {
    p->tbuf = work;
    p->tbuf_owned = false;
  }
  return MK_OK;
}

extern "C" int mk_filt_plan_set_halve(mk_filt_plan* p, int halve_edges) {
  MK_REQUIRE(p, MK_ERR_ARG, "null plan");
  for (auto& s : p->h_segs) s.flags = halve_edges ? 1 : 0;
  return upload(p);
}

// ---------------------------------------------------------------------------
// Stand-alone DCT-I (Bluestein), rows of one length n.

namespace {
// Workspace of the general path (power-of-two P): descriptors, chirp
// spectrum, rows.
int64_t dct1_general_bytes(int64_t nrow, int64_t n, int elem_bytes) {
  Geometry g = geometry(2 * (n - 1) + 1, elem_bytes);
  return (nrow * g.P + g.P) * 2 * elem_bytes + 4096;
}
// Column count of the 2^11-row path for FP64 rows of n points (0: general
// path), and its workspace: descriptors, chirp spectrum, rows, twiddle
// tables, chirp.
int dct1_q1(int64_t n, int elem_bytes) {
  const int64_t need = 2 * (n - 1) + 1;
  return elem_bytes == 8 && need > kHotP2 && !getenv("MK_FFT_NO_HOT") ? q1_at_least(need) : 0;
}
int64_t dct1_rows_bytes(int64_t nrow, int64_t n, int q) {
  return ((nrow + 1) * q * kHotP2 + kTwCommon + q1_table_elems(q) + n) * 16 + 4096;
}
}  // namespace

extern "C" int64_t mk_dct1_workspace_bytes(int64_t nrow, int64_t n, int elem_bytes) {
  if (n < 2 || nrow < 0 || (elem_bytes != 4 && elem_bytes != 8)) return -1;
  const int q = dct1_q1(n, elem_bytes);
  return q ? dct1_rows_bytes(nrow, n, q) : dct1_general_bytes(nrow, n, elem_bytes);
}

namespace {
// FP64 rows through the 2^11-row engine: P = 2^11 q >= 2m+1 points (a
// power of two on the general path, 1.4 times as many on average), the chirp
// from a table built once per call.
int dct1_rows64(const double* x, double* y, int64_t nrow, int64_t n, int q, void* work, hipStream_t st) {
  unsigned char* w = (unsigned char*)work;
  const int64_t P = (int64_t)q * kHotP2;
  cx<double>* V = (cx<double>*)(w + 4096);
  cx<double>* tb = V + P;
  cx<double>* tw = tb + nrow * P;
  cx<double>* qt = tw + kTwCommon;
  cx<double>* chirp = qt + q1_table_elems(q);
  Seg s[2] = {};
  s[0].in_stride = s[0].out_stride = n;
  s[0].t_stride = P;
  s[0].s_ptr = V;
  s[0].tw_off = kTwCommon;
  s[0].rows = (int32_t)nrow;
  s[0].n = (int32_t)n;
  s[0].per2 = (q + 1) / 2;
  s[0].q1 = q;
  s[1] = s[0];
  s[1].rows = 1;
  const int64_t nb = col_blocks<double>(q);
  MK_REQUIRE(nrow * nb < INT32_MAX && nrow * s[0].per2 < INT32_MAX, MK_ERR_ARG, "too many rows");
  Seg* d = (Seg*)w;
  static_assert(2 * sizeof(Seg) <= 4096, "descriptors");
  MK_HIP(hipMemcpyAsync(d, s, sizeof(s), hipMemcpyHostToDevice, st));
  MK_HIP(hipStreamSynchronize(st));
  launch_col_tables<double>(q, tw, qt, st);
  launch_chirp(chirp, n, st);
  const cx<double>* ct = qt + (int64_t)q * kRowTw;
  launch_cols_fwd<double>(q, kBSpec, d + 1, 1, nb, x, V, tw, ct, chirp, 0, st);
  launch_rows<double>(kBSpec, d + 1, 1, s[0].per2, V, tw, 0, false, st);
  launch_cols_fwd<double>(q, kBlue, d, 1, nrow * nb, x, tb, tw, ct, chirp, 0, st);
  launch_rows<double>(kBlue, d, 1, nrow * s[0].per2, tb, tw, 0, false, st);
  launch_cols_inv<double>(q, kBlue, d, 1, nrow * nb, tb, y, tw, ct, chirp, st);
  return mk::check_launch("dct1");
}

template <typename T, typename TIO>
int dct1_impl(const TIO* x, TIO* y, int64_t nrow, int64_t n, void* work, int64_t work_bytes, void* stream) {
  MK_REQUIRE(nrow >= 0 && n >= 2, MK_ERR_ARG, "DCT-I needs n >= 2 (got %lld)", (long long)n);
  if (nrow == 0) return MK_OK;
  MK_REQUIRE(x && y && work, MK_ERR_ARG, "null argument");
  MK_REQUIRE(n < (int64_t(1) << 30) && nrow < INT32_MAX, MK_ERR_ARG, "DCT-I of %lld rows of %lld points is too large",
             (long long)nrow, (long long)n);
  // the 2^11-row path wants slightly more than the general one where P is
  // about the same; a caller's workspace of the general size is still served
  const int q = dct1_q1(n, sizeof(T));
  const bool rows = q && work_bytes >= dct1_rows_bytes(nrow, n, q);
  const int64_t need = dct1_general_bytes(nrow, n, sizeof(T));
  MK_REQUIRE(rows || work_bytes >= need, MK_ERR_ARG, "workspace too small (%lld < %lld)", (long long)work_bytes,
             (long long)need);
  MK_REQUIRE(((uintptr_t)work & 255) == 0, MK_ERR_ARG, "workspace must be 256-byte aligned");
  allow_lds_all();
  hipStream_t st = mk::as_stream(stream);
  if constexpr (sizeof(T) == 8) {
    if (rows) return dct1_rows64(x, y, nrow, n, q, work, st);
  }
  int64_t desc[6] = {nrow, n, 0, n, 0, n};
  std::vector<Seg> segs;
  int64_t n1, n2, te, se;
  size_t l1, l2;
  int r = build_segs(1, desc, sizeof(T), false, segs, &n1, &n2, &te, &se, &l1, &l2);
  if (r) return r;
  MK_REQUIRE(n1 < INT32_MAX && n2 < INT32_MAX, MK_ERR_ARG, "too many rows");
  // workspace: [segment descriptor (aligned)] [V spectrum P] [T buffer nrow*P]
  unsigned char* w = (unsigned char*)work;
  Seg* d_seg = (Seg*)w;
  cx<T>* V = (cx<T>*)(w + 4096);
  cx<T>* tb = V + segs[0].t_stride;
  Seg s0 = segs[0];
  s0.s_off = 0;
  s0.s_ptr = V;
  MK_HIP(hipMemcpyAsync(d_seg, &s0, sizeof(Seg), hipMemcpyHostToDevice, st));
  MK_HIP(hipStreamSynchronize(st));
  // spectrum of the conjugate chirp: a one-row pass (rows = 1) over the same geometry
  Seg sv = s0;
  sv.rows = 1;
  Seg* d_sv = d_seg + 1;
  MK_HIP(hipMemcpyAsync(d_sv, &sv, sizeof(Seg), hipMemcpyHostToDevice, st));
  MK_HIP(hipStreamSynchronize(st));
  k1_kernel<T, TIO, kBSpec><<<(unsigned)s0.per1, kThreads, l1, st>>>(d_sv, 1, x, V);
  k2_kernel<T, T, kBSpec><<<(unsigned)s0.per2, kThreads, l2, st>>>(d_sv, 1, V);
  k1_kernel<T, TIO, kBlue><<<(unsigned)n1, kThreads, l1, st>>>(d_seg, 1, x, tb);
  k2_kernel<T, T, kBlue><<<(unsigned)n2, kThreads, l2, st>>>(d_seg, 1, tb);
  k3_kernel<T, TIO, kBlue><<<(unsigned)n1, kThreads, l1, st>>>(d_seg, 1, tb, y);
  return mk::check_launch("dct1");
}
}  // namespace

// Static workspace of mk_dct1_f64_noalloc: the Bluestein workspace (segment
// descriptors, chirp spectrum, nrow x P complex FP64 rows) for callers that
// cannot allocate device memory.  64 MiB per device that runs the library,
// held until the process ends.  Host code never uses this name as an
// address: it asks hipGetSymbolAddress for each device's copy once, with
// that device current, and passes that pointer on.
constexpr int64_t kScratchBytes = int64_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The current device's address of `scratch` (looked up on its first use).
int scratch_ptr(void** out) {
  int dev = -1;
  MK_HIP(hipGetDevice(&dev));
  MK_REQUIRE(dev >= 0 && dev < kMaxDevices, MK_ERR_ARG, "device index %d outside 0..%d", dev, kMaxDevices - 1);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    MK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    MK_REQUIRE(p != nullptr && ((uintptr_t)p & 255) == 0, MK_ERR_HIP, "scratch address lookup gave %p", p);
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return MK_OK;
}
}  // namespace

extern "C" int mk_dct1_f64_noalloc(const double* x, double* y, int64_t nrow, int64_t n, void* stream) {
  MK_REQUIRE(nrow >= 0 && n >= 2, MK_ERR_ARG, "DCT-I needs nrow >= 0 and n >= 2 (got %lld, %lld)", (long long)nrow,
             (long long)n);
  if (nrow == 0) return MK_OK;
  MK_REQUIRE(n < (int64_t(1) << 30), MK_ERR_ARG, "DCT-I of %lld points is too long", (long long)n);
  const int64_t q = dct1_q1(n, 8);
  int64_t need = dct1_general_bytes(nrow, n, 8);
  if (q) need = std::min(need, dct1_rows_bytes(nrow, n, (int)q));
  MK_REQUIRE(need > 0 && need <= kScratchBytes, MK_ERR_ARG,
             "mk_dct1_f64_noalloc: %lld rows of %lld points need %lld B of workspace, more than its %lld B static "
             "scratch; use mk_dct1_f64 with a caller workspace (or fewer rows per call)",
             (long long)nrow, (long long)n, (long long)need, (long long)kScratchBytes);
  void* ws = nullptr;
  int r = scratch_ptr(&ws);
  if (r) return r;
  return dct1_impl<double, double>(x, y, nrow, n, ws, kScratchBytes, stream);
}

extern "C" int mk_dct1_f64(const double* x, double* y, int64_t nrow, int64_t n, void* work, int64_t work_bytes,
                           void* stream) {
  return dct1_impl<double, double>(x, y, nrow, n, work, work_bytes, stream);
}
extern "C" int mk_dct1_f32(const float* x, float* y, int64_t nrow, int64_t n, void* work, int64_t work_bytes,
                           void* stream) {
  return dct1_impl<float, float>(x, y, nrow, n, work, work_bytes, stream);
}
