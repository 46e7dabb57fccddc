// device.hpp -- device-side building blocks shared by the line kernels:
// complex arithmetic, power-of-two butterflies, the kernel argument
// block and the load/store helpers.
#pragma once

#include "lines.hpp"
#include "rfh.hpp"

namespace rfh {
namespace dev {

// ------------------------------------------------------------ complex math

template <typename T>
struct alignas(2 * sizeof(T)) C2 {
  T x, y;
};

template <typename T>
__device__ __forceinline__ C2<T> operator+(C2<T> a, C2<T> b) {
  return {a.x + b.x, a.y + b.y};
}
template <typename T>
__device__ __forceinline__ C2<T> operator-(C2<T> a, C2<T> b) {
  return {a.x - b.x, a.y - b.y};
}
template <typename T>
__device__ __forceinline__ C2<T> operator*(T s, C2<T> a) {
  return {s * a.x, s * a.y};
}
template <typename T>
__device__ __forceinline__ C2<T> cmul(C2<T> a, C2<T> b) {
  return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename T>
__device__ __forceinline__ C2<T> conjc(C2<T> a) {
  return {a.x, -a.y};
}
// a * (dir * i)
template <typename T>
__device__ __forceinline__ C2<T> rot(C2<T> a, T dir) {
  return {-dir * a.y, dir * a.x};
}
// w, conjugated when dir > 0 (tables hold forward-sign roots)
template <typename T>
__device__ __forceinline__ C2<T> dirw(C2<T> w, T dir) {
  return {w.x, dir < T(0) ? w.y : -w.y};
}

// Tile index of this workgroup with XCD-contiguous placement.  The
// dispatcher deals workgroups round-robin to the 8 XCDs (workgroup i runs on
// XCD i mod 8); renumbering them so that each XCD owns one contiguous run of
// tiles keeps the cache lines that neighbouring tiles share inside one L2.
__device__ __forceinline__ unsigned xcd_tile() {
  constexpr unsigned kXcd = 8;
  const unsigned g = gridDim.x, i = blockIdx.x;
  if (g < 2 * kXcd) return i;
  const unsigned x = i % kXcd, k = i / kXcd, q = g / kXcd, r = g % kXcd;
  return x * q + (x < r ? x : r) + k;
}

// q = u / d for 0 <= u < 2^22 via a float reciprocal and one correction.
__device__ __forceinline__ int fdiv(int u, int d, float inv) {
  int q = int(float(u) * inv);
  const int r = u - __mul24(q, d);
  q += (r >= d) - (r < 0);
  return q;
}

// -------------------------------------------------------------- butterflies
// dir = -1: X_k = sum_m v_m e^{-2 pi i m k / R}; dir = +1 the conjugate kernel.

template <typename T>
__device__ __forceinline__ void dft2(C2<T> *v) {
  const C2<T> a = v[0];
  v[0] = a + v[1];
  v[1] = a - v[1];
}

template <typename T>
__device__ __forceinline__ void dft4(C2<T> *v, T dir) {
  const C2<T> t0 = v[0] + v[2], t1 = v[0] - v[2], t2 = v[1] + v[3];
  const C2<T> t3 = rot(v[1] - v[3], dir);
  v[0] = t0 + t2;
  v[2] = t0 - t2;
  v[1] = t1 + t3;
  v[3] = t1 - t3;
}

template <typename T>
__device__ __forceinline__ void dft8(C2<T> *v, T dir) {
  C2<T> e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
  dft4(e, dir);
  dft4(o, dir);
  const T s = T(0.707106781186547524400844362104849039);
  const C2<T> o1 = {s * (o[1].x - dir * o[1].y), s * (o[1].y + dir * o[1].x)};
  const C2<T> o2 = rot(o[2], dir);
  const C2<T> o3 = {s * (-o[3].x - dir * o[3].y), s * (-o[3].y + dir * o[3].x)};
  v[0] = e[0] + o[0];
  v[4] = e[0] - o[0];
  v[1] = e[1] + o1;
  v[5] = e[1] - o1;
  v[2] = e[2] + o2;
  v[6] = e[2] - o2;
  v[3] = e[3] + o3;
  v[7] = e[3] - o3;
}

template <typename T>
__device__ __forceinline__ void dft16(C2<T> *v, T dir) {
  C2<T> e[8], o[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    e[k] = v[2 * k];
    o[k] = v[2 * k + 1];
  }
  dft8(e, dir);
  dft8(o, dir);
  const T c1 = T(0.923879532511286756128183189396788933);
  const T s1 = T(0.382683432365089771728459984030398866);
  const T r = T(0.707106781186547524400844362104849039);
  const T cs[8] = {T(1), c1, r, s1, T(0), -s1, -r, -c1};
  const T sn[8] = {T(0), s1, r, c1, T(1), c1, r, s1};
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const C2<T> w = {cs[k], dir * sn[k]};
    const C2<T> t = cmul(o[k], w);
    v[k] = e[k] + t;
    v[k + 8] = e[k] - t;
  }
}

template <int R, typename T>
__device__ __forceinline__ void dft(C2<T> *v, T dir) {
  static_assert(R == 2 || R == 4 || R == 8 || R == 16, "power-of-two radices");
  if constexpr (R == 2) dft2(v);
  else if constexpr (R == 4) dft4(v, dir);
  else if constexpr (R == 8) dft8(v, dir);
  else dft16(v, dir);
}

// ----------------------------------------------------------- line kernel

enum LineOp {
  OP_C2C = 0,     // plain complex lines
  OP_PASSA = 1,   // four-step pass A (columns), inter-pass twiddle on store
  OP_PASSB = 2,   // four-step pass B (rows)
  OP_BLUE = 3,    // Bluestein entirely in LDS
  OP_R2C_EVEN = 4,
  OP_R2C_ODD = 5,
  OP_C2R_EVEN = 6,
  OP_C2R_ODD = 7,
  OP_R2R = 8,     // real line -> pre_elem -> FFT -> post_elem (DCT/DST, Hartley, FFTPACK)
  // elementwise passes of the multi-pass Bluestein form (no FFT; count = other)
  OP_BLUE_IN = 11,   // work[m] = x[m] * conj(chirp[m]) for m < n, zero up to bn2
  OP_BLUE_MUL = 12,  // work[m] *= kernel[m]
  OP_BLUE_OUT = 13,  // y[m] = fct * work[m] * conj(chirp[m]) for m < n
  // Bluestein rows of the three-pass form: forward FFT of the row, times the
  // kernel (t2, laid out by rows: bin k of row aux at aux * n + k), inverse FFT,
  // times the inverse four-step twiddle (tables t0 / t1); written back in place
  OP_BLUEROW = 14,
};
// OP_R2R packs its modes into LineArgs::sub
constexpr int R2R_ORTHO = 1 << 16, R2R_CONJ = 1 << 17, R2R_FLIP = 1 << 18;
constexpr int R2R_SINCOS = 1 << 19;  // the factors are computed, there is no table
enum SubFlags {
  SUB_CHIRP = 1,   // pass A: multiply loads by the chirp, zero beyond n
  SUB_FINAL = 4,   // pass A: multiply by the chirp and fct, keep m = aux + k other < n
  SUB_CONJ = 8,    // Bluestein backward / r2c conj output / c2r conj input
};

template <typename T>
struct LineArgs {
  int64_t nlines;
  int nb;
  int64_t bdim[kMaxBatchDims], bsi[kMaxBatchDims], bso[kMaxBatchDims];
  int64_t esi, eso;
  const T *in;
  T *out;
  int nin, nout, lfast_in, lfast_out;
  int auxdim;    // batch dim whose index is a line's aux (four-step row / column)
  int twlds_lo, twlds_hi;  // pass A of the specialised kernel: four-step twiddle
                           // tables (t0 / t1 entries) copied to LDS; 0 = read globally
  FftDesc f;
  const C2<T> *tw, *gen;
  T dir, fct;
  int sub;
  int64_t bign;  // n of the transform (Bluestein / real), N of a four-step
  int64_t other; // four-step: N2 in pass A, N1 in pass B
  int shift;
  const C2<T> *t0, *t1, *t2;  // op tables
  int rot_in, rot_out;  // element-index rotations of the line set (0: none)
  int op;
};

// (j + r) mod n for 0 <= j, r < n
__device__ __forceinline__ int rot_index(int j, int r, int n) {
  const int q = j + r;
  return q >= n ? q - n : q;
}

// Bluestein column passes (chirped loads of pass A, final stores of pass C):
// element j of column aux is element m = j other + aux of the transform
// line; with the line rotated by rot it is read from / written to element
// (m + rot) mod n, which lies (that - aux) line elements (es / other scalars
// each) from the column's start.  Offset in scalars from the column start.
__device__ __forceinline__ int64_t blue_col_offset(int j, int64_t m, int rot, int64_t n,
                                                   int aux, int64_t es, int64_t other) {
  if (!rot) return int64_t(j) * es;
  int64_t q = m + rot;
  if (q >= n) q -= n;
  return (q - aux) * (es / other);
}

template <bool V, typename T>
__device__ __forceinline__ C2<T> ldc(const T *p) {
  if constexpr (V) return *reinterpret_cast<const C2<T> *>(p);
  else return C2<T>{p[0], p[1]};
}
template <bool V, typename T>
__device__ __forceinline__ void stc(T *p, C2<T> v) {
  if constexpr (V) *reinterpret_cast<C2<T> *>(p) = v;
  else {
    p[0] = v.x;
    p[1] = v.y;
  }
}

template <typename T>
__device__ __forceinline__ C2<T> big_twiddle(const LineArgs<T> &a, int64_t e) {
  const int64_t mask = (int64_t(1) << a.shift) - 1;
  return cmul(a.t0[e & mask], a.t1[e >> a.shift]);
}

// e^{i pi num/den}: integer argument reduction, then sincospi in the
// working precision (FP64 for complex128, FP32 for complex64).
template <typename T>
__device__ __forceinline__ C2<T> expipi(int64_t num, int64_t den) {
  const int64_t per = 2 * den;
  int64_t r = num % per;
  if (r < 0) r += per;
  if constexpr (sizeof(T) == 8) {
    double s, c;
    sincospi(double(r) / double(den), &s, &c);
    return C2<T>{T(c), T(s)};
  } else {
    float s, c;
    sincospif(float(double(r) / double(den)), &s, &c);
    return C2<T>{c, s};
  }
}

// e^{i pi num / 4n}, num >= 0: computed, or from a table of the plan's (num
// <= 2n).  The DCT / DST factors e^{i pi j / 2n} and e^{i pi (2j + 1) / 4n}.
template <typename T>
struct ComputedRoot {
  int64_t n;
  __device__ __forceinline__ C2<T> operator()(int64_t num) const { return expipi<T>(num, 4 * n); }
};
template <typename T>
struct TableRoot {
  const C2<T> *t;
  __device__ __forceinline__ C2<T> operator()(int num) const { return t[num]; }
};

// Element j of the complex work line built from input line x (element
// stride es) for the real-transform modes of PreMode; m = work length.  I: the
// type of indices within a line.
template <typename T, typename I, typename Rt>
__device__ __forceinline__ C2<T> pre_elem(int mode, const T *x, int64_t es, I n, I m, I j,
                                          bool ortho, bool conj, bool flip, const Rt &root) {
  const T sqrt2 = T(1.41421356237309504880168872420969808);
  C2<T> v = {T(0), T(0)};
  switch (mode) {
    case kPreRealAsComplex:
      if (j < n) {
        T xv = x[j * es];
        if (flip && j >= 2 && (j % 2) == 0) xv = -xv;
        v.x = xv;
      }
      break;
    case kPreHermitian: {  // half complex input X[0..n/2]
      const I h = n / 2;
      if (j == 0) {
        v = C2<T>{x[0], T(0)};
      } else if (j < n - h || (2 * j < n)) {
        v = C2<T>{x[j * es], x[j * es + 1]};
        if (conj) v.y = -v.y;
      } else if (2 * j == n) {
        v = C2<T>{x[j * es], T(0)};
      } else {
        const I k = n - j;
        v = C2<T>{x[k * es], x[k * es + 1]};
        if (!conj) v.y = -v.y;
      }
      break;
    }
    case kPreDct1: {
      const I src = j < n ? j : m - j;
      T xv = x[src * es];
      if (ortho && (src == 0 || src == n - 1)) xv *= sqrt2;
      v.x = xv;
      break;
    }
    case kPreDst1:
      if (j >= 1 && j <= n) v.x = x[(j - 1) * es];
      else if (j >= n + 2) v.x = -x[(m - 1 - j) * es];
      break;
    case kPreType2:
      if (j < n) v.x = x[j * es];
      break;
    case kPreDct3:
      if (j < n) {
        T xv = x[j * es];
        if (j == 0 && ortho) xv *= sqrt2;
        const T w = j == 0 ? T(1) : T(2);
        v = (w * xv) * root(2 * j);
      }
      break;
    case kPreDst3:
      if (j >= 1 && j <= n) {
        T xv = x[(j - 1) * es];
        if (j == 1 && ortho) xv *= sqrt2;
        const T w = j == n ? T(1) : T(2);
        v = (w * xv) * root(2 * j);
      }
      break;
    case kPreType4:
      if (j < n) v = x[j * es] * conjc(root(2 * j));
      break;
    case kPreHalfcomplex: {
      if (j == 0) {
        v.x = x[0];
      } else if (2 * j < n) {
        v = C2<T>{x[(2 * j - 1) * es], x[(2 * j) * es]};
        if (conj) v.y = -v.y;
      } else if (2 * j == n) {
        v.x = x[(n - 1) * es];
      } else {
        const I k = n - j;
        v = C2<T>{x[(2 * k - 1) * es], -x[(2 * k) * es]};
        if (conj) v.y = -v.y;
      }
      break;
    }
    case kPreRealPairs:
      if (2 * j < n) v = C2<T>{x[2 * j * es], x[(2 * j + 1) * es]};
      break;
    case kPreDct2N:
    case kPreDst2N: {
      // v_j = x_2j for 2j < n, v_{n-1-j} = x_2j+1: V = FFT_n(v) gives
      // DCT-II_k = 2 Re(e^{-i pi k/2n} V_k); DST-II is DCT-II of (-1)^j x_j
      // read backwards
      const I i = 2 * j < n ? 2 * j : 2 * (n - 1 - j) + 1;
      T xv = x[i * es];
      if (mode == kPreDst2N && (i & 1)) xv = -xv;
      v.x = xv;
      break;
    }
    case kPreDct3N:
    case kPreDst3N: {
      // a = x (DCT-III) or x reversed (DST-III), a_n = 0, ortho scales x_0 by
      // sqrt 2; V_j = (a_j - i a_{n-j}) e^{i pi j/2n} and the inverse FFT of
      // length n holds the even outputs up and the odd outputs down
      auto at = [&](I q) -> T {  // (the load has no condition around it)
        const I qc = q < n ? q : n - 1, src = mode == kPreDct3N ? qc : n - 1 - qc;
        T xv = x[src * es];
        if (ortho && src == 0) xv *= sqrt2;
        return q < n ? xv : T(0);
      };
      v = cmul(C2<T>{at(j), -at(n - j)}, root(2 * j));
      break;
    }
    case kPreHalfSpectrum: {
      // z_j = Σ_k [A_k + i e^{2πik/n} D_k] e^{2πikj/(n/2)} with A = X_k + conj X_{h-k},
      // D = X_k - conj X_{h-k}: the inverse FFT of length h = n/2 gives
      // y_2j + i y_2j+1.  Imaginary parts of bins 0 and h are ignored.
      const I h = n / 2;
      C2<T> xj = {x[j * es], x[j * es + 1]}, xm = {x[(h - j) * es], x[(h - j) * es + 1]};
      if (conj) {
        xj.y = -xj.y;
        xm.y = -xm.y;
      }
      if (j == 0) {
        xj.y = T(0);
        xm.y = T(0);
      }
      const C2<T> A = xj + conjc(xm);
      const C2<T> B = cmul(xj - conjc(xm), expipi<T>(2 * j, n));
      v = C2<T>{A.x - B.y, A.y + B.x};
      break;
    }
  }
  return v;
}

// r2c bin k (0..n/2) of a real line of even length n from the length-n/2
// spectrum Z of its pairs z_j = x_2j + i x_2j+1 (get(q) = Z_q):
// X_k = (Z_k + conj Z_{h-k}) / 2 + e^{-2πik/n} (Z_k - conj Z_{h-k}) / 2i.
template <typename T, typename G>
__device__ __forceinline__ C2<T> half_spectrum_bin(G &&get, int64_t n, int64_t k) {
  const int64_t h = n / 2;
  if (k == 0 || k == h) {
    const C2<T> z = get(0);
    return C2<T>{k == 0 ? z.x + z.y : z.x - z.y, T(0)};
  }
  const C2<T> zk = get(k), zm = conjc(get(h - k));
  const C2<T> fe = T(0.5) * (zk + zm);
  const C2<T> dd = zk - zm;
  const C2<T> fo = C2<T>{T(0.5) * dd.y, T(-0.5) * dd.x};
  return fe + cmul(expipi<T>(-2 * k, n), fo);
}

// Real output element k from the transformed work line (get(q) = bin q)
// for the PostMode modes other than kPostComplexHalf; fct not applied.
template <typename T, typename I, typename G, typename Rt>
__device__ __forceinline__ T post_elem(int mode, G &&get, I n, I k, bool ortho, bool flip,
                                       const Rt &root) {
  const T isqrt2 = T(0.707106781186547524400844362104849039);
  T r = T(0);
  switch (mode) {
    case kPostReal:
      r = get(k).x;
      if (flip && k >= 2 && (k % 2) == 0) r = -r;
      break;
    case kPostDct1:
      r = get(k).x;
      if (ortho && (k == 0 || k == n - 1)) r *= isqrt2;
      break;
    case kPostDst1:
      r = -get(k + 1).y;
      break;
    case kPostDct2: {
      const C2<T> z = cmul(get(k), conjc(root(2 * k)));
      r = T(2) * z.x;
      if (ortho && k == 0) r *= isqrt2;
      break;
    }
    case kPostDst2: {
      const C2<T> z = cmul(get(k + 1), conjc(root(2 * (k + 1))));
      r = -T(2) * z.y;
      if (ortho && k == 0) r *= isqrt2;
      break;
    }
    case kPostDct3:
      r = get(k).x;
      break;
    case kPostDst3:
      r = get(k).y;
      break;
    case kPostDct4:
    case kPostDst4: {
      const C2<T> z = cmul(get(k), conjc(root(2 * k + 1)));
      r = mode == kPostDct4 ? T(2) * z.x : -T(2) * z.y;
      break;
    }
    case kPostHartley:
      r = get(k).x + get(k).y;
      break;
    case kPostPackHalfcomplex:  // (the forward sign rule flips inputs only)
      if (k == 0) r = get(0).x;
      else if (k % 2) r = get((k + 1) / 2).x;
      else r = get(k / 2).y;
      break;
    case kPostRealPairs:
      r = (k % 2) ? get(k / 2).y : get(k / 2).x;
      break;
    case kPostDct2N:
    case kPostDst2N: {
      const I q = mode == kPostDct2N ? k : n - 1 - k;
      const C2<T> z = cmul(get(q), conjc(root(2 * q)));
      r = T(2) * z.x;
      if (ortho && k == 0) r *= isqrt2;
      break;
    }
    case kPostDct3N:
    case kPostDst3N:
      r = get((k % 2 == 0) ? k / 2 : n - 1 - (k - 1) / 2).x;
      if (mode == kPostDst3N && (k & 1)) r = -r;
      break;
  }
  return r;
}

}  // namespace dev

// Compile-time specialised kernels (fast.hip); false when none matches.
template <typename T>
bool launch_fast(int op, const dev::LineArgs<T> &a, bool lf_in, bool lf_out, bool vin,
                 bool vout, hipStream_t s);
extern bool g_fast_enabled;

// Persistent software-pipelined FP32 passes of the complex64 1024 x 1024
// four-step plans (pass1024.hip); false when the pass does not match.
bool launch_pass1024(int op, const dev::LineArgs<float> &a, bool lf_in, bool lf_out, bool vin,
                     bool vout, hipStream_t s);

// Persistent software-pipelined FP32 transform of contiguous complex64 lines
// of 4096 (pipe4096.hip); false when the pass does not match.
bool launch_pipe4096(int op, const dev::LineArgs<float> &a, bool lf_in, bool lf_out, bool vin,
                     bool vout, hipStream_t s);

// Split-precision MFMA kernels (mfma.hip): the kernel family launched, or
// nullptr when the mode is off or the pass has no matrix-core form
// (contiguous complex64 lines of 4096, the 1024-point four-step passes).
const char *launch_mfma(int op, const dev::LineArgs<float> &a, bool lf_in, bool lf_out,
                        bool vin, bool vout, hipStream_t s);
void mfma_probe(int bf, const float *a, const float *b, float *d, hipStream_t s);
extern int g_precision_mode;
// launches of the matrix-core kernels in precision mode `mode` (0: all modes)
uint64_t mfma_launch_count(int mode);
// while on (per thread), a missing operand table is an error instead of an
// allocation
void mfma_no_alloc(bool on);
// the FP64-derived DFT-16 operand table of a mode and direction (host only)
int mfma_operand_table(int mode, int dir, float *out, int cap);

}  // namespace rfh
