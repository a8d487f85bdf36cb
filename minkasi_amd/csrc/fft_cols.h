// Column passes of the 2^11-point-row FFT engine, instantiated per precision
// by fft_cols_f32.hip and fft_cols_f64.hip.
//
// A workgroup takes CW adjacent columns of one row of the batch; thread
// (c, b) does butterfly b of column c.  The first radix-R1 stage reads global
// memory straight into registers and the last radix-R2 stage writes it
// straight from them, so a column transform of up to 256 points has one LDS
// exchange (none up to 16 points).  In the LDS tile point e of column c lies
// at e CW + c: lanes are consecutive columns, without bank conflicts.
//
// Bound: HBM.  The filter's forward pass reads n reals and writes P complex
// per row (P about n), its inverse pass reads P complex and writes n reals:
// 54 and 46 us for 215 rows of 100003 samples (0.26 GB each, 4.9 and 5.7 TB/s
// with part of it in the last-level cache).  Passes over the 1.5 times longer
// even extension, each stage through LDS, took 138 and 86 us.
#pragma once
#include "fft_engine.h"

namespace mkfft {
namespace {

__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float buf_load(__amdgpu_buffer_rsrc_t r, uint32_t off, float) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0u, 0));
}
__device__ __forceinline__ double buf_load(__amdgpu_buffer_rsrc_t r, uint32_t off, double) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0u, 0));
}

// The filter's placement of a row in the L = 2P real points: sample s at
// index s - c0 mod L, c0 = ceil(m/2), with the two end samples halved.  With
// P >= m+1 the samples fill index [0, P/2) and [3P/2, 2P) only, so the middle
// half of every column is zero.
//
// First the row's ends are brought to zero: q = a0 + a1 cos(pi s / m) with
// q(0) = y_0, q(m) = y_m is subtracted, and its image l0 a0 + l1 a1 cos(...)
// (both terms are eigenvectors of C W C, l0 and l1 stored behind the row's
// spectra) is added to the output; cos(pi s / m) is the real part of
// exp(i pi (2 col + w + c0) / m) exp(i pi (s - 2 col - w - c0) / m), a factor
// per column and one per time row, from a table per row length.  Without it the zero padding cuts a red
// row off at its ends, and the rounding of the large spectrum that makes,
// weighted by W, is 1.2 to 1.4 times the error of the even extension's
// transform; with it 0.6 to 1.1 times (rows of random walk plus white noise,
// 10^4 to 2.6 10^5 samples).
template <typename T, typename TIO, int Q>
__global__ void __launch_bounds__(col_threads<T>(Q)) cols_fwd_kernel(const Seg* __restrict__ segs, int nseg, int mode,
                                                                     const void* __restrict__ in,
                                                                     cx<T>* __restrict__ tbuf,
                                                                     const cx<T>* __restrict__ tw,
                                                                     const cx<T>* __restrict__ coltw,
                                                                     const cx<T>* __restrict__ chirp, int comp,
                                                                     int64_t nblk) {
  constexpr int R1 = col_r1(Q), R2 = col_r2(Q), CW = col_cw<T>(Q);
  constexpr int64_t P = (int64_t)Q * kRowLen;
  extern __shared__ unsigned char smem_raw[];
  cx<T>* buf = reinterpret_cast<cx<T>*>(smem_raw);  // [Q][CW]
  // XCD-aware order: the pieces of one row run on one XCD, so the cache lines
  // that neighbouring pieces share are fetched once
  const int64_t per = ((int64_t)gridDim.x + 7) / 8;
  const int64_t bid = (int64_t)(blockIdx.x % 8) * per + blockIdx.x / 8;
  if (bid >= nblk) return;
  const Seg& sg = segs[find_seg(segs, nseg, bid, 1)];
  const int local = (int)(bid - sg.base1);
  const int row = local / (kRowLen / CW), col0 = (local % (kRowLen / CW)) * CW;
  const int m = sg.n - 1;
  const int c = threadIdx.x % CW;
  int b = threadIdx.x / CW;
  if (CW % 64 == 0) b = __builtin_amdgcn_readfirstlane(b);
  const int col = col0 + c;
  cx<T>* trow = tbuf + sg.t_off + (int64_t)row * sg.t_stride;
  cx<T> v[R1];
  if (b < R2) {
    if (mode == kFilter) {
      const TIO* x = reinterpret_cast<const TIO*>(in) + sg.in_off + (int64_t)row * sg.in_stride;
      const __amdgpu_buffer_rsrc_t xrs = row_rsrc(x, (uint32_t)(m + 1) * (uint32_t)sizeof(TIO));
      const cx<T>* em = tw + sg.em_off;
      const cx<T> z0 = em[2 * col], z1 = em[2 * col + 1];
      const T a0 = T(0.5) * (T)x[0] + T(0.5) * (T)x[m], a1 = T(0.5) * (T)x[0] - T(0.5) * (T)x[m];
      if (col0 == 0 && threadIdx.x == 0) {
        const gptr<const T> lam = as_global<const T>(sg.s_ptr) + (int64_t)row * sg.s_stride + 2 * (P + 1);
        tbuf[sg.e_off + row] = {lam[0] * a0, lam[1] * a1};
      }
      const int c0 = (m + 1) >> 1;
      const int s0 = 2 * (kRowLen * b + col) + c0;  // sample of element r = 0
#pragma unroll
      for (int r = 0; r < R1; r++) {
        if (4 * r >= R1 && 4 * (r + 1) <= 3 * R1) {  // the zero half
          v[r] = {T(0), T(0)};
          continue;
        }
        // samples outside [0, m] give offsets past the row's bytes, which
        // read as zero (a negative one wraps to a large offset)
        const int s = s0 + 2 * kRowLen * R2 * r - (2 * r >= R1 ? (int)(2 * P) : 0);
        uint32_t o0 = (uint32_t)s * (uint32_t)sizeof(TIO), o1 = (uint32_t)(s + 1) * (uint32_t)sizeof(TIO);
        asm("" : "+v"(o1));  // keeps the second offset from becoming "first + immediate", which does not wrap
        const T x0 = (T)buf_load(xrs, o0, TIO(0)), x1 = (T)buf_load(xrs, o1, TIO(0));
        const cx<T> e = cscale(em[2 * kRowLen + b + R2 * r], a1);
        v[r].re = (uint32_t)s <= (uint32_t)m ? x0 - (a0 + (e.re * z0.re - e.im * z0.im)) : T(0);
        v[r].im = (uint32_t)(s + 1) <= (uint32_t)m ? x1 - (a0 + (e.re * z1.re - e.im * z1.im)) : T(0);
      }
      // the end samples' columns: index 2P - c0 (sample 0) and m - c0
      const int e0 = (int)(((2 * P - c0) >> 1) & (kRowLen - 1)), e1 = ((m - c0) >> 1) & (kRowLen - 1);
      if ((e0 >= col0 && e0 < col0 + CW) || (e1 >= col0 && e1 < col0 + CW)) {  // uniform
#pragma unroll
        for (int r = 0; r < R1; r++) {
          const int s = s0 + 2 * kRowLen * R2 * r - (2 * r >= R1 ? (int)(2 * P) : 0);
          if (s == 0 || s == m) v[r].re *= T(0.5);
          if (s + 1 == 0 || s + 1 == m) v[r].im *= T(0.5);
        }
      }
    } else if constexpr (sizeof(T) == 8) {
      const double* x = reinterpret_cast<const double*>(in) + sg.in_off + (int64_t)row * sg.in_stride;
      if (mode == kFSpec) {
        // lag |i| (i mod L) of the kernel: h, or h reversed about m/2
#pragma unroll
        for (int r = 0; r < R1; r++) {
          const int64_t i = 2 * ((int64_t)kRowLen * (b + R2 * r) + col);
          T e[2];
#pragma unroll
          for (int w = 0; w < 2; w++) {
            const int64_t a = i + w <= P ? i + w : 2 * P - (i + w);
            e[w] = a <= m ? (T)x[comp ? m - a : a] : T(0);
          }
          v[r] = {e[0], e[1]};
        }
      } else {
        const int64_t N = 2 * (int64_t)m;
#pragma unroll
        for (int r = 0; r < R1; r++) {
          const int64_t j = (int64_t)kRowLen * (b + R2 * r) + col;
          v[r] = {T(0), T(0)};
          if (mode == kBlue) {
            if (j <= m) {
              const T wgt = (j == 0 || j == m) ? T(1) : T(2);
              const cx<T> ch = chirp ? chirp[j] : expmi<T>((j * j) % (2 * N), N);
              v[r] = cscale(ch, wgt * (T)x[j]);
            }
          } else {  // kBSpec: conj(chirp) at lags -m..m, placed mod P
            const int64_t t = j <= m ? j : (j >= P - m ? P - j : -1);
            if (t >= 0) v[r] = cconj(chirp ? chirp[t] : expmi<T>((t * t) % (2 * N), N));
          }
        }
      }
    }
    dft_small<T, false, R1>(v);
    if constexpr (R2 == 1) {
#pragma unroll
      for (int r = 0; r < R1; r++) trow[(int64_t)r * kRowLen + col] = v[r];
    } else {
#pragma unroll
      for (int r = 0; r < R1; r++) buf[(b * R1 + r) * CW + c] = v[r];
    }
  }
  if constexpr (R2 > 1) {
    __syncthreads();
    if (b < R1) {
      cx<T> u[R2];
#pragma unroll
      for (int r = 0; r < R2; r++) u[r] = buf[(b + r * R1) * CW + c];
#pragma unroll
      for (int r = 1; r < R2; r++) u[r] = cmul(u[r], coltw[b * r]);
      dft_small<T, false, R2>(u);
#pragma unroll
      for (int r = 0; r < R2; r++) trow[(int64_t)(b + r * R1) * kRowLen + col] = u[r];
    }
  }
}

// Two reals at any element alignment.
template <typename T>
struct __attribute__((packed, aligned(sizeof(T)))) Pair {
  T a, b;
};

template <typename T, typename TIO, int Q>
__global__ void __launch_bounds__(col_threads<T>(Q)) cols_inv_kernel(const Seg* __restrict__ segs, int nseg, int mode,
                                                                     const cx<T>* __restrict__ tbuf,
                                                                     void* __restrict__ out,
                                                                     const cx<T>* __restrict__ tw,
                                                                     const cx<T>* __restrict__ coltw,
                                                                     const cx<T>* __restrict__ chirp) {
  constexpr int R1 = col_r1(Q), R2 = col_r2(Q), CW = col_cw<T>(Q);
  constexpr int64_t P = (int64_t)Q * kRowLen;
  extern __shared__ unsigned char smem_raw[];
  cx<T>* buf = reinterpret_cast<cx<T>*>(smem_raw);  // [Q][CW]
  const Seg& sg = segs[find_seg(segs, nseg, blockIdx.x, 3)];
  const int local = (int)((int64_t)blockIdx.x - sg.base3);
  const int row = local / (kRowLen / CW), col0 = (local % (kRowLen / CW)) * CW;
  const int m = sg.n - 1;
  const int c = threadIdx.x % CW;
  int b = threadIdx.x / CW;
  if (CW % 64 == 0) b = __builtin_amdgcn_readfirstlane(b);
  const int col = col0 + c;
  const cx<T>* trow = tbuf + sg.t_off + (int64_t)row * sg.t_stride;
  constexpr int RL = R2 > 1 ? R2 : R1;  // radix of the last stage
  cx<T> u[RL];
  if constexpr (R2 == 1) {
#pragma unroll
    for (int r = 0; r < R1; r++) u[r] = trow[(int64_t)r * kRowLen + col];
    dft_small<T, true, R1>(u);
  } else {
    if (b < R2) {
      cx<T> v[R1];
#pragma unroll
      for (int r = 0; r < R1; r++) v[r] = trow[(int64_t)(b + r * R2) * kRowLen + col];
      dft_small<T, true, R1>(v);
#pragma unroll
      for (int r = 0; r < R1; r++) buf[(b * R1 + r) * CW + c] = v[r];
    }
    __syncthreads();
    if (b >= R1) return;
#pragma unroll
    for (int r = 0; r < R2; r++) u[r] = buf[(b + r * R1) * CW + c];
#pragma unroll
    for (int r = 1; r < R2; r++) u[r] = cmul(u[r], cconj(coltw[b * r]));
    dft_small<T, true, R2>(u);
  }
  // time row j1 = b + r R1 of the tile (r, when one stage does it all)
  constexpr int STEP = R2 > 1 ? R1 : 1;
  TIO* y = reinterpret_cast<TIO*>(out) + sg.out_off + (int64_t)row * sg.out_stride;
  if (mode == kFilter) {
    const T scale = T(0.25) / (T)P;  // 1/P of the inverse transform, 1/4 of the packing (row pass)
    const cx<T>* em = tw + sg.em_off;
    const cx<T> z0 = em[2 * col], z1 = em[2 * col + 1];
    const cx<T> q = tbuf[sg.e_off + row];  // the end modes' image
    const int c0 = (m + 1) >> 1;
    const int e0 = (int)(((2 * P - c0) >> 1) & (kRowLen - 1)), e1 = ((m - c0) >> 1) & (kRowLen - 1);
    const bool ends = (sg.flags & 1) && ((e0 >= col0 && e0 < col0 + CW) || (e1 >= col0 && e1 < col0 + CW));
#pragma unroll
    for (int r = 0; r < RL; r++) {
      if (4 * r >= RL && 4 * (r + 1) <= 3 * RL) continue;  // the half no sample lies in
      const int j1 = b + r * STEP;
      const int s = 2 * (kRowLen * j1 + col) + c0 - (2 * r >= RL ? (int)(2 * P) : 0);
      const cx<T> e = cscale(em[2 * kRowLen + j1], q.im);
      T o0 = u[r].re * scale + (q.re + (e.re * z0.re - e.im * z0.im));
      T o1 = u[r].im * scale + (q.re + (e.re * z1.re - e.im * z1.im));
      if (ends) {
        if (s == 0 || s == m) o0 *= T(0.5);
        if (s + 1 == 0 || s + 1 == m) o1 *= T(0.5);
      }
      if (s >= 0 && s < m) {
        *reinterpret_cast<Pair<TIO>*>(y + s) = {(TIO)o0, (TIO)o1};
      } else {
        if (s == m) y[s] = (TIO)o0;
        if (s == -1) y[0] = (TIO)o1;
      }
    }
  } else if constexpr (sizeof(T) == 8) {  // kBlue
    const T scale = T(1) / (T)P;
    const int64_t N = 2 * (int64_t)m;
#pragma unroll
    for (int r = 0; r < RL; r++) {
      const int64_t k = (int64_t)kRowLen * (b + r * STEP) + col;
      if (k <= m) {
        const cx<T> w = cscale(u[r], scale);
        const cx<T> ch = chirp ? chirp[k] : expmi<T>((k * k) % (2 * N), N);
        y[k] = (TIO)(ch.re * w.re - ch.im * w.im);
      }
    }
  }
}

template <typename T, int I = 0>
void fwd_by_index(int idx, int mode, const Seg* segs, int nseg, int64_t nblk, const void* in, cx<T>* tbuf,
                  const cx<T>* tw, const cx<T>* coltw, const cx<T>* chirp, int comp, hipStream_t st) {
  if constexpr (I < kNumQ1) {
    constexpr int Q = kQ1[I];
    if (idx != I) return fwd_by_index<T, I + 1>(idx, mode, segs, nseg, nblk, in, tbuf, tw, coltw, chirp, comp, st);
    cols_fwd_kernel<T, T, Q><<<(unsigned)(mk::cdiv(nblk, 8) * 8), col_threads<T>(Q), col_lds<T>(Q), st>>>(
        segs, nseg, mode, in, tbuf, tw, coltw, chirp, comp, nblk);
  }
}
template <typename T, int I = 0>
void inv_by_index(int idx, int mode, const Seg* segs, int nseg, int64_t nblk, const cx<T>* tbuf, void* out,
                  const cx<T>* tw, const cx<T>* coltw, const cx<T>* chirp, hipStream_t st) {
  if constexpr (I < kNumQ1) {
    constexpr int Q = kQ1[I];
    if (idx != I) return inv_by_index<T, I + 1>(idx, mode, segs, nseg, nblk, tbuf, out, tw, coltw, chirp, st);
    cols_inv_kernel<T, T, Q><<<(unsigned)nblk, col_threads<T>(Q), col_lds<T>(Q), st>>>(segs, nseg, mode, tbuf, out, tw,
                                                                                      coltw, chirp);
  }
}

}  // namespace

template <typename T>
void launch_cols_fwd(int q, int mode, const Seg* segs, int nseg, int64_t nblk, const void* in, cx<T>* tbuf,
                     const cx<T>* tw, const cx<T>* coltw, const cx<T>* chirp, int comp, hipStream_t st) {
  fwd_by_index<T>(q1_index(q), mode, segs, nseg, nblk, in, tbuf, tw, coltw, chirp, comp, st);
}
template <typename T>
void launch_cols_inv(int q, int mode, const Seg* segs, int nseg, int64_t nblk, const cx<T>* tbuf, void* out,
                     const cx<T>* tw, const cx<T>* coltw, const cx<T>* chirp, hipStream_t st) {
  inv_by_index<T>(q1_index(q), mode, segs, nseg, nblk, tbuf, out, tw, coltw, chirp, st);
}

}  // namespace mkfft
