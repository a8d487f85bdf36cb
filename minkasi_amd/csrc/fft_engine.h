// Shared pieces of the FFT kernels: complex arithmetic, in-register DFTs,
// the segment descriptor, and the column / row passes of the 2^11-point-row
// engine (fft_cols_*.hip, fft_rows.hip), which fft.hip plans and launches.
#pragma once
#include "common.h"

namespace mkfft {

template <typename T>
struct alignas(2 * sizeof(T)) cx {
  T re, im;
};
template <typename T>
__device__ __forceinline__ cx<T> cadd(cx<T> a, cx<T> b) { return {a.re + b.re, a.im + b.im}; }
template <typename T>
__device__ __forceinline__ cx<T> csub(cx<T> a, cx<T> b) { return {a.re - b.re, a.im - b.im}; }
template <typename T>
__device__ __forceinline__ cx<T> cmul(cx<T> a, cx<T> b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <typename T>
__device__ __forceinline__ cx<T> cconj(cx<T> a) { return {a.re, -a.im}; }
template <typename T>
__device__ __forceinline__ cx<T> cscale(cx<T> a, T s) { return {a.re * s, a.im * s}; }

__device__ __forceinline__ void sincospi_t(float x, float* s, float* c) { sincospif(x, s, c); }
__device__ __forceinline__ void sincospi_t(double x, double* s, double* c) { sincospi(x, s, c); }

// exp(-i*pi*num/den) for integers 0 <= num < 2*den.
template <typename T>
__device__ __forceinline__ cx<T> expmi(int64_t num, int64_t den) {
  T s, c;
  sincospi_t((T)(-(double)num / (double)den), &s, &c);
  return {c, s};
}

// ---- In-register DFTs (natural order in and out) ----------------------------
template <typename T, bool INV>
__device__ __forceinline__ void dft2(cx<T>* v) {
  cx<T> a = v[0], b = v[1];
  v[0] = cadd(a, b);
  v[1] = csub(a, b);
}
template <typename T, bool INV>
__device__ __forceinline__ void dft4(cx<T>& a0, cx<T>& a1, cx<T>& a2, cx<T>& a3) {
  cx<T> b0 = cadd(a0, a2), b1 = csub(a0, a2), b2 = cadd(a1, a3), d = csub(a1, a3);
  cx<T> b3 = INV ? cx<T>{-d.im, d.re} : cx<T>{d.im, -d.re};  // (+/-i) * d
  a0 = cadd(b0, b2);
  a2 = csub(b0, b2);
  a1 = cadd(b1, b3);
  a3 = csub(b1, b3);
}
template <typename T, bool INV>
__device__ __forceinline__ void dft4v(cx<T>* v) { dft4<T, INV>(v[0], v[1], v[2], v[3]); }
template <typename T, bool INV>
__device__ __forceinline__ void dft8(cx<T>* v) {
  const T c = T(0.70710678118654752440);
  cx<T> e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
  cx<T> o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
  dft4<T, INV>(e0, e1, e2, e3);
  dft4<T, INV>(o0, o1, o2, o3);
  if (!INV) {
    o1 = {c * (o1.re + o1.im), c * (o1.im - o1.re)};   // * exp(-i pi/4)
    o2 = {o2.im, -o2.re};                               // * -i
    o3 = {c * (o3.im - o3.re), -c * (o3.re + o3.im)};  // * exp(-3i pi/4)
  } else {
    o1 = {c * (o1.re - o1.im), c * (o1.re + o1.im)};   // * exp(i pi/4)
    o2 = {-o2.im, o2.re};                               // * i
    o3 = {-c * (o3.re + o3.im), c * (o3.re - o3.im)};  // * exp(3i pi/4)
  }
  v[0] = cadd(e0, o0); v[4] = csub(e0, o0);
  v[1] = cadd(e1, o1); v[5] = csub(e1, o1);
  v[2] = cadd(e2, o2); v[6] = csub(e2, o2);
  v[3] = cadd(e3, o3); v[7] = csub(e3, o3);
}
template <typename T, bool INV>
__device__ __forceinline__ void dft3(cx<T>* v) {
  const T h = T(0.86602540378443864676);  // sin(2 pi / 3)
  cx<T> a = cadd(v[1], v[2]), d = csub(v[1], v[2]);
  cx<T> t = {v[0].re - T(0.5) * a.re, v[0].im - T(0.5) * a.im};
  cx<T> u = INV ? cx<T>{-h * d.im, h * d.re} : cx<T>{h * d.im, -h * d.re};  // (+/-i) sin(2pi/3) d
  v[0] = cadd(v[0], a);
  v[1] = cadd(t, u);
  v[2] = csub(t, u);
}
template <typename T, bool INV>
__device__ __forceinline__ void dft5(cx<T>* v) {
  const T c1 = T(0.30901699437494742410), c2 = T(-0.80901699437494742410);  // cos(2pi/5), cos(4pi/5)
  const T s1 = T(0.95105651629515357212), s2 = T(0.58778525229247312917);   // sin(2pi/5), sin(4pi/5)
  cx<T> a1 = cadd(v[1], v[4]), b1 = csub(v[1], v[4]), a2 = cadd(v[2], v[3]), b2 = csub(v[2], v[3]);
  cx<T> t1 = {v[0].re + c1 * a1.re + c2 * a2.re, v[0].im + c1 * a1.im + c2 * a2.im};
  cx<T> t2 = {v[0].re + c2 * a1.re + c1 * a2.re, v[0].im + c2 * a1.im + c1 * a2.im};
  cx<T> u1 = {s1 * b1.re + s2 * b2.re, s1 * b1.im + s2 * b2.im};
  cx<T> u2 = {s2 * b1.re - s1 * b2.re, s2 * b1.im - s1 * b2.im};
  // forward: y1 = t1 - i u1, y4 = t1 + i u1, y2 = t2 - i u2, y3 = t2 + i u2
  cx<T> iu1 = INV ? cx<T>{-u1.im, u1.re} : cx<T>{u1.im, -u1.re};
  cx<T> iu2 = INV ? cx<T>{-u2.im, u2.re} : cx<T>{u2.im, -u2.re};
  v[0] = cadd(v[0], cadd(a1, a2));
  v[1] = cadd(t1, iu1);
  v[4] = csub(t1, iu1);
  v[2] = cadd(t2, iu2);
  v[3] = csub(t2, iu2);
}

// cos and sin of 2 pi e / N for the composite sizes with internal twiddles.
constexpr double kCos9[9] = {1.0, 0.76604444311897803520, 0.17364817766693034885, -0.5, -0.93969262078590838405,
                             -0.93969262078590838405, -0.5, 0.17364817766693034885, 0.76604444311897803520};
constexpr double kSin9[9] = {0.0, 0.64278760968653932632, 0.98480775301220805937, 0.86602540378443864676,
                             0.34202014332566873304, -0.34202014332566873304, -0.86602540378443864676,
                             -0.98480775301220805937, -0.64278760968653932632};
constexpr double kC16 = 0.92387953251128675613, kS16 = 0.38268343236508977173, kR2 = 0.70710678118654752440;
constexpr double kCos16[16] = {1.0, kC16, kR2, kS16, 0.0, -kS16, -kR2, -kC16, -1.0, -kC16, -kR2, -kS16, 0.0, kS16, kR2, kC16};
constexpr double kSin16[16] = {0.0, kS16, kR2, kC16, 1.0, kC16, kR2, kS16, 0.0, -kS16, -kR2, -kC16, -1.0, -kC16, -kR2, -kS16};

// v * exp(-/+ 2 pi i e / 16), e a compile-time constant after unrolling.
template <typename T, bool INV>
__device__ __forceinline__ cx<T> mul_w16(cx<T> v, int e) {
  if (e == 0) return v;
  if (e == 8) return {-v.re, -v.im};
  if (e == 4) return INV ? cx<T>{-v.im, v.re} : cx<T>{v.im, -v.re};
  if (e == 12) return INV ? cx<T>{v.im, -v.re} : cx<T>{-v.im, v.re};
  const T c = (T)kCos16[e], s = (T)(INV ? kSin16[e] : -kSin16[e]);
  if (e == 2 || e == 6 || e == 10 || e == 14) {
    // |c| == |s|: two products of sums
    const T r = (T)kR2;
    const T sc = kCos16[e] > 0 ? r : -r;
    const bool same = (kCos16[e] > 0) == ((INV ? kSin16[e] : -kSin16[e]) > 0);
    return same ? cx<T>{sc * (v.re - v.im), sc * (v.im + v.re)} : cx<T>{sc * (v.re + v.im), sc * (v.im - v.re)};
  }
  return cmul(v, cx<T>{c, s});
}
template <typename T, bool INV>
__device__ __forceinline__ cx<T> mul_w9(cx<T> v, int e) {
  if (e == 0) return v;
  return cmul(v, cx<T>{(T)kCos9[e], (T)(INV ? kSin9[e] : -kSin9[e])});
}

constexpr int mod_inv(int a, int b) {  // a^-1 mod b
  for (int i = 1; i < b; i++)
    if (a * i % b == 1) return i;
  return 1;
}

template <typename T, bool INV, int R>
__device__ __forceinline__ void dft_small(cx<T>* v);

// N = A B with A, B coprime (Good-Thomas: no internal twiddles).
template <typename T, bool INV, int A, int B>
__device__ __forceinline__ void dft_pfa(cx<T>* v) {
  constexpr int N = A * B, KA = B * mod_inv(B % A, A), KB = A * mod_inv(A % B, B);
  cx<T> t[N];
#pragma unroll
  for (int n2 = 0; n2 < B; n2++) {
    cx<T> u[A];
#pragma unroll
    for (int n1 = 0; n1 < A; n1++) u[n1] = v[(B * n1 + A * n2) % N];
    dft_small<T, INV, A>(u);
#pragma unroll
    for (int k1 = 0; k1 < A; k1++) t[k1 * B + n2] = u[k1];
  }
#pragma unroll
  for (int k1 = 0; k1 < A; k1++) {
    cx<T> u[B];
#pragma unroll
    for (int n2 = 0; n2 < B; n2++) u[n2] = t[k1 * B + n2];
    dft_small<T, INV, B>(u);
#pragma unroll
    for (int k2 = 0; k2 < B; k2++) v[(KA * k1 + KB * k2) % N] = u[k2];
  }
}

// N = A A (9 = 3 3, 16 = 4 4): x[n1 A + n2], twiddle w_N^(n2 k1), X[k1 + A k2].
template <typename T, bool INV, int A>
__device__ __forceinline__ void dft_sq(cx<T>* v) {
  constexpr int N = A * A;
  cx<T> t[N];
#pragma unroll
  for (int n2 = 0; n2 < A; n2++) {
    cx<T> u[A];
#pragma unroll
    for (int n1 = 0; n1 < A; n1++) u[n1] = v[n1 * A + n2];
    dft_small<T, INV, A>(u);
#pragma unroll
    for (int k1 = 0; k1 < A; k1++)
      t[k1 * A + n2] = N == 16 ? mul_w16<T, INV>(u[k1], n2 * k1) : mul_w9<T, INV>(u[k1], n2 * k1);
  }
#pragma unroll
  for (int k1 = 0; k1 < A; k1++) {
    cx<T> u[A];
#pragma unroll
    for (int n2 = 0; n2 < A; n2++) u[n2] = t[k1 * A + n2];
    dft_small<T, INV, A>(u);
#pragma unroll
    for (int k2 = 0; k2 < A; k2++) v[k1 + A * k2] = u[k2];
  }
}

template <typename T, bool INV, int R>
__device__ __forceinline__ void dft_small(cx<T>* v) {
  if constexpr (R == 2) dft2<T, INV>(v);
  else if constexpr (R == 3) dft3<T, INV>(v);
  else if constexpr (R == 4) dft4v<T, INV>(v);
  else if constexpr (R == 5) dft5<T, INV>(v);
  else if constexpr (R == 6) dft_pfa<T, INV, 2, 3>(v);
  else if constexpr (R == 8) dft8<T, INV>(v);
  else if constexpr (R == 9) dft_sq<T, INV, 3>(v);
  else if constexpr (R == 10) dft_pfa<T, INV, 2, 5>(v);
  else if constexpr (R == 12) dft_pfa<T, INV, 4, 3>(v);
  else if constexpr (R == 15) dft_pfa<T, INV, 3, 5>(v);
  else if constexpr (R == 16) dft_sq<T, INV, 4>(v);
  else static_assert(R == 1, "unsupported radix");
}

// ---- Segments ----------------------------------------------------------------
// A segment: `rows` rows sharing one length n and one plan.
struct Seg {
  int64_t in_off, in_stride;    // input rows (elements of the input type)
  int64_t out_off, out_stride;  // output rows
  int64_t t_off, t_stride;      // T buffer rows (complex)
  int64_t s_off, s_stride;      // spectrum rows (reals; general path: P+1, 2^11-row path: 2 (P+2); Bluestein: stride 0)
  void* s_ptr;                  // device address of this segment's spectrum rows (set at upload)
  // 2^11-row path: in the twiddle table this column count's row twiddles and
  // this row length's end-mode phases; in the T buffer the rows' end-mode
  // outputs
  int64_t tw_off, em_off, e_off;
  int32_t rows, n, l1, l2, cw, flags;  // l1 = log2(P1), or -1 when P1 is not a power of two
  int64_t base1, base2, base3;  // first global item of K1, K2, K3
  int32_t per1, per2;           // items per row for K1/K3, K2
  int32_t r2, p1;               // k1 values per K2 item; column length P1 (2^a 3^b 5^c)
  int32_t q1, hot;              // 2^11-row path: the transform's column count; whether the segment takes that path
};

// A pointer read from memory is generic to the compiler (flat loads, which
// also wait on the LDS counter); this one is known to be global.
template <typename X>
using gptr = __attribute__((address_space(1))) X*;
template <typename X>
__device__ __forceinline__ gptr<X> as_global(void* p) {
  return (gptr<X>)(uintptr_t)p;
}

enum Mode { kFilter = 0, kFSpec = 1, kBlue = 2, kBSpec = 3 };

__device__ inline int find_seg(const Seg* segs, int nseg, int64_t g, int which) {
  int lo = 0, hi = nseg - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    int64_t b = which == 1 ? segs[mid].base1 : (which == 2 ? segs[mid].base2 : segs[mid].base3);
    if (b <= g) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// ---- The 2^11-point-row engine -------------------------------------------------
// P = Q1 * 2^11 complex points, j = 2^11 j1 + j2 in time, k = k1 + Q1 k2 in
// frequency.  Column pass: Q1-point DFTs down the columns (no twiddles);
// row pass: 2^11-point DFTs along the rows with the four-step twiddle
// w_P^(k1 j2) folded into the row transform's own twiddles.
constexpr int kRowL2 = 11;
constexpr int kRowLen = 1 << kRowL2;
constexpr int kRowThreads = 256;

// Column counts: at most two radices of {2..6, 8, 9, 10, 12, 15, 16}, so a
// column pass needs at most one LDS exchange.  The steps between them cost at
// most 25 % of padding (5 % on average for TODs of 10^4 to 2 10^5 samples).
constexpr int kQ1[] = {2,  3,  4,  5,  6,  8,  9,  10, 12, 15,  16,  18,  20,  24,  27,  30,  32,  36,  40,  45, 48,
                       50, 54, 60, 64, 72, 80, 90, 96, 100, 108, 120, 128, 144, 150, 160, 180, 192, 225, 240, 256};
constexpr int kNumQ1 = sizeof(kQ1) / sizeof(kQ1[0]);
constexpr bool is_radix(int r) {
  return (r >= 2 && r <= 6) || r == 8 || r == 9 || r == 10 || r == 12 || r == 15 || r == 16;
}
// First radix of a Q1-point column transform: Q1 itself up to 16, else the
// smaller factor of the most balanced split (equal radices leave no thread
// idle in either stage), with a multiple of four first where there is a
// choice (its elements that lie in the zero half of the input are known).
constexpr int col_r1(int q) {
  if (q <= 16 && is_radix(q)) return q;
  int best = 0;
  for (int r = 2; r <= 16; r++)
    if (is_radix(r) && q % r == 0 && is_radix(q / r) && r * r <= q) best = r;
  if (best % 4 != 0 && (q / best) % 4 == 0) return q / best;
  return best;
}
constexpr int col_r2(int q) { return q / col_r1(q); }
constexpr bool all_q1_split() {
  for (int i = 0; i < kNumQ1; i++)
    if (col_r1(kQ1[i]) == 0 || col_r1(kQ1[i]) * col_r2(kQ1[i]) != kQ1[i]) return false;
  return true;
}
static_assert(all_q1_split(), "a column count does not split into two radices");

// Columns per workgroup and its threads: one thread per (column, butterfly).
// 64 columns make a wave share one butterfly (uniform twiddles, 512-byte
// runs); 32 or 16 where more would take over 64 KiB of LDS.
template <typename T>
constexpr int col_cw(int q) {
  if (col_r2(q) == 1) return 256;
  int cw = 64;
  while (cw * q * 2 * (int)sizeof(T) > 65536) cw /= 2;
  return cw;
}
template <typename T>
constexpr int col_threads(int q) {
  const int nb = col_r1(q) > col_r2(q) ? col_r1(q) : col_r2(q);
  return col_r2(q) == 1 ? 256 : (col_cw<T>(q) * nb + 63) / 64 * 64;
}
template <typename T>
constexpr int col_lds(int q) {
  return col_r2(q) == 1 ? 0 : col_cw<T>(q) * q * 2 * (int)sizeof(T);
}
inline int q1_index(int q) {
  for (int i = 0; i < kNumQ1; i++)
    if (kQ1[i] == q) return i;
  return -1;
}
// The smallest column count with 2^11 q >= points (0: none).
inline int q1_at_least(int64_t points) {
  for (int i = 0; i < kNumQ1; i++)
    if ((int64_t)kQ1[i] * kRowLen >= points) return kQ1[i];
  return 0;
}

// Twiddle tables (built in FP64, stored in T):
//   common: w_256^(k r) at [r 16 + k] (r, k < 16), w_2048^(k r) at
//           [256 + r 256 + k] (r < 8, k < 256), w_4096^k at [2304 + k] (k < 256);
//   per column count: rows of kRowTw entries per k1: w_(16 Q1)^(k1 r) (16),
//           w_(256 Q1)^(k1 r) (16), w_P^(k1 r) (8), w_2P^k1; then Q1 entries w_Q1^e.
constexpr int kTwCommon = 256 + 8 * 256 + 256;
constexpr int kRowTw = 48;
inline int64_t q1_table_elems(int q) { return (int64_t)q * (kRowTw + 1); }

// Launchers (fft_cols_f32.hip, fft_cols_f64.hip, fft_rows.hip).  tw: the
// twiddle tables, coltw: the column count's w_Q1^e; comp: which kernel
// spectrum of the filter (0: h, 1: its reversal); chirp: Bluestein's
// exp(-i pi j^2 / N), j <= m, or null to evaluate it per element.
template <typename T>
void launch_col_tables(int q, cx<T>* common, cx<T>* tab, hipStream_t st);
template <typename T>
void launch_cols_fwd(int q, int mode, const Seg* segs, int nseg, int64_t nblk, const void* in, cx<T>* tbuf,
                     const cx<T>* tw, const cx<T>* coltw, const cx<T>* chirp, int comp, hipStream_t st);
template <typename T>
void launch_cols_inv(int q, int mode, const Seg* segs, int nseg, int64_t nblk, const cx<T>* tbuf, void* out,
                     const cx<T>* tw, const cx<T>* coltw, const cx<T>* chirp, hipStream_t st);
// spec32: FSpec stores FP32 spectra from the FP64 transform.
template <typename T>
void launch_rows(int mode, const Seg* segs, int nseg, int64_t nblk, cx<T>* tbuf, const cx<T>* tw, int comp,
                 bool spec32, hipStream_t st);
// Lets the row pass use more than 64 KiB of LDS (once, before any launch that
// may be captured).
void allow_rows_lds();
constexpr int end_phase_elems(int q) { return 2 * kRowLen + q; }
template <typename T>
void launch_end_phases(cx<T>* out, int64_t n, int q, hipStream_t st);
// The filter's eigenvalues of each row's two end modes (after the spectra).
void launch_end_modes(const Seg* segs, int nseg, int64_t rows, const double* h, bool spec32, hipStream_t st);
void launch_chirp(cx<double>* chirp, int64_t n, hipStream_t st);
// Column-pass workgroups per row.
template <typename T>
inline int col_blocks(int q) { return kRowLen / col_cw<T>(q); }

}  // namespace mkfft
