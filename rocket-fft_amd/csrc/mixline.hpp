// mixline.hpp -- the general line kernel: a group of L lines of any length
// whose stages run out of ONE line buffer per line in LDS.
//
// Each thread owns one place j of one line and holds the elements of its
// butterflies of a stage in registers (at most kMaxElems of them: one
// butterfly of a large radix, several of a small one): a stage reads its
// inputs from LDS, waits until every thread has read, and writes its outputs
// over them.  One buffer instead of two ping-pong buffers is half the LDS per
// line, so twice the lines (waves) are resident per CU, and a thread's place
// in its line is found once instead of per butterfly and stage.  The radices
// (2 .. 17, gpu_radices) are chosen so that a stage's butterflies fill the
// line's threads: 1000 = 10 x 10 x 10 is three stages of 100 threads.
//
// Layout between stages.  After the stage of radix R whose predecessors
// multiply to ns, the line is N / (ns R) blocks of ns R elements; block q
// starts at q P with a pitch P >= ns R chosen (block_pitch) so that the
// stage's writes (runs of ns elements, P apart) spread over the LDS banks.
// The next stage reads element j + r N/R' of the line at
// (j / ns') P + j mod ns' + r (N/R'/ns') P: padding changes only the strides.
//
// Direction.  Every stage runs the forward transform; an inverse transform
// exchanges real and imaginary parts as elements are loaded and stored.
//
// Bluestein (OP_BLUE, OP_BLUEROW).  The last forward stage holds bins
// j + r N/R in registers, which are the inputs of the first stage of the
// inverse transform run backwards (each stage undone in reverse order:
// butterfly, conjugate twiddles, write to where the forward stage had read).
// So the kernel product happens in registers between two butterflies, and the
// inverse transform needs no tables of its own: S - 1 exchanges each way.
#pragma once

#include <type_traits>

#include "butterfly.hpp"
#include "mixgeom.hpp"

namespace rfh {

namespace dev {

template <typename T>
constexpr int kMaxElems = mix_max_elems(sizeof(T) == 8);
template <typename T>
constexpr int kMixThreads = mix_max_threads(sizeof(T) == 8);

// OP of a kernel that runs every operation but the real-to-real ones, by
// LineArgs::op (the batch executor's).  Lines are loaded to LDS and stored from
// LDS by one loop per operation, and the stages exist once per radix: with each
// operation's loads and stores unrolled into each radix, as in k_lines, the
// kernel took 1.9 MB of code and 400 s to compile, at the same speed (1447 and
// 1452 us on the 4096-job batch; 188 KB and 19 s this way).
constexpr int OP_ANY = -1;
template <int OP, typename T>
__device__ __forceinline__ int op_of(const LineArgs<T> &a) {
  return OP == OP_ANY ? a.op : OP;
}
constexpr bool real_in(int op) { return op == OP_R2C_EVEN || op == OP_R2C_ODD || op == OP_R2R; }
constexpr bool real_out(int op) { return op == OP_C2R_EVEN || op == OP_C2R_ODD || op == OP_R2R; }
// factors e^{i pi q / 4n} of a real-to-real line
template <bool SINCOS, typename T>
__device__ __forceinline__ auto root_of(const LineArgs<T> &a) {
  if constexpr (SINCOS) return ComputedRoot<T>{a.bign};
  else return TableRoot<T>{a.t0};
}
// Forms of the kernel beside the general one: lines of at most one butterfly of
// a small radix (short_lines), without the other radices' registers; groups of
// short contiguous lines that move flat (Walk); lines with a prime above 17 of
// more than kFewPairs output pairs a thread, whose sums take registers; real-to-
// real lines without a table of their factors.
constexpr int kShort = 1, kFlat = 2, kPrime = 4, kSinCos = 8;
// operations that have a flat form
constexpr bool is_flat_op(int op) {
  return op == OP_C2C || op == OP_R2C_EVEN || op == OP_R2C_ODD || op == OP_C2R_EVEN ||
         op == OP_C2R_ODD || op == OP_R2R;
}
constexpr bool is_blue_op(int op) { return op == OP_BLUE || op == OP_BLUEROW; }
__device__ __forceinline__ bool is_blue(int op) { return is_blue_op(op); }
// whether an op stores bin by bin, straight from the last stage's registers
__device__ __forceinline__ bool elem_store(int op) { return op != OP_R2C_EVEN && op != OP_R2R; }

template <typename T>
struct MixCtx {
  const T *in;  // this thread's line in global memory
  T *out;
  C2<T> *ln;    // ... and in LDS
  int aux;      // index along the line set's auxdim (four-step row / column)
  int j;        // place in the line
  bool ok;      // the line exists and the thread has a place in it
  bool line;    // ... the line exists (a line alone in its group: for every thread)
  const T *in0;  // the group's first line, its lines and their LDS (FLAT only)
  T *out0;
  int nl;
  C2<T> *lds;
};

// How the threads walk `count` elements of each line: those of a line by its
// own threads; a line alone in its group takes all of the group's threads, also
// those without a place in the stages; FLAT: the group's lines one after
// another, neighbours to neighbouring threads, whichever line they are in.
template <typename T, int FORM>
struct Walk {
  static constexpr bool FLAT = (FORM & kFlat) != 0, SHORT = (FORM & kShort) != 0;
  const MixGeom &m;
  const MixCtx<T> &c;
  int first, step, total, count;
  float inv;
  bool on;
  __device__ __forceinline__ Walk(const MixGeom &m_, const MixCtx<T> &c_, int count_)
      : m(m_),
        c(c_),
        first(FLAT ? int(threadIdx.x) : c.j),
        step(FLAT || (!SHORT && m.L == 1) ? int(blockDim.x) : m.T),
        total(FLAT ? c.nl * count_ : count_),
        count(count_),
        inv(1.0f / float(count_)),
        on(FLAT || (!SHORT && m.L == 1 ? c.line : c.ok)) {}
  // element e's index in its line; the line's addresses
  __device__ __forceinline__ int place(int e, MixCtx<T> &at) const {
    at = c;
    if (!FLAT) return e;
    const int l = fdiv(e, count, inv);
    at.in = c.in0 + unsigned(__mul24(l, m.flat_in));
    at.out = c.out0 + unsigned(__mul24(l, m.flat_out));
    at.ln = c.lds + __mul24(l, m.ld);
    return e - __mul24(l, count);
  }
};

template <typename T>
__device__ __forceinline__ C2<T> swapri(C2<T> a, bool sw) {
  return sw ? C2<T>{a.y, a.x} : a;
}

// Complex elements at any scalar-aligned address: a global access of two
// (or four) dwords needs dword alignment only.
template <typename T>
struct __attribute__((packed, aligned(sizeof(T)))) PackedC2 {
  T x, y;
};
template <typename T>
__device__ __forceinline__ C2<T> gload(const T *p) {
  const PackedC2<T> v = *reinterpret_cast<const PackedC2<T> *>(p);
  return C2<T>{v.x, v.y};
}
template <typename T>
__device__ __forceinline__ void gstore(T *p, C2<T> v) {
  *reinterpret_cast<PackedC2<T> *>(p) = PackedC2<T>{v.x, v.y};
}

// W_N^e from the half-size tables
template <typename T>
__device__ __forceinline__ C2<T> step_twiddle(const LineArgs<T> &a, int k, int aux) {
  const uint64_t e = uint64_t(unsigned(k)) * uint64_t(unsigned(aux));
  const unsigned mask = (1u << a.shift) - 1u;
  return cmul(a.t0[unsigned(e) & mask], a.t1[e >> a.shift]);
}

// Factors (chirps, four-step twiddles) a thread holds beside its elements: all R
// of them took registers that a kernel of every radix spilled (four-step columns
// 203 complex64 and 433 complex128 ones, Bluestein lines 40 and 649): us, all /
// these, 2000 lines of 30000 complex64 673 / 592, 64 of 10^6 907 / 801, 400
// columns of 30000 129 / 113, 256 lines of 4099 complex128 51.9 / 40.6.
template <typename T, int OP, int R>
constexpr int kFactors = OP == OP_ANY ? R : (sizeof(T) == 8 ? 4 : 8);

// The element stride of a line that moves flat: 24-bit products (flat_lines).
struct Stride24 {
  int v;
  __device__ __forceinline__ explicit Stride24(int64_t s) : v(int(s)) {}
  __device__ __forceinline__ operator int() const { return v; }
};
__device__ __forceinline__ int operator*(int i, Stride24 s) { return __mul24(i, s.v); }

// Inputs j + r NR (r < R) of a line, with the op's pre-processing.  CLAMP:
// beyond the line its last element instead.  FLAT: 24-bit strides.
template <typename T, int OP, int R, bool CLAMP = false, bool FLAT = false>
__device__ __forceinline__ void op_load(const LineArgs<T> &a, const MixCtx<T> &c, int j, int NR,
                                        C2<T> *v) {
  constexpr int S = kFactors<T, OP, R>;
  const bool cj = (a.sub & SUB_CONJ) != 0;
  using Es = std::conditional_t<FLAT, Stride24, int64_t>;
  const Es es = Es(a.esi);
  const int op = op_of<OP>(a);
  auto at = [&](int r) { return CLAMP ? min(j + r * NR, a.f.n - 1) : j + r * NR; };
  if (op == OP_C2C || op == OP_PASSB || op == OP_BLUEROW || op == OP_PASSA) {
    if (op == OP_PASSA && (a.sub & SUB_CHIRP)) {  // x[m] conj(chirp[m]), zero from m = n on
      // (loads without a condition around them, so that all are in flight)
#pragma unroll
      for (int s = 0; s < R; s += S) {
        C2<T> w[S];
#pragma unroll
        for (int r = s; r < R && r < s + S; ++r) {
          const int64_t m = int64_t(at(r)) * a.other + c.aux;
          const int jj = m < a.bign ? at(r) : 0;
          const int64_t mc = m < a.bign ? m : c.aux;
          w[r - s] = a.t2[mc];
          v[r] = gload(c.in + blue_col_offset(jj, mc, a.rot_in, a.bign, c.aux, es, a.other));
        }
#pragma unroll
        for (int r = s; r < R && r < s + S; ++r) {
          const bool on = int64_t(at(r)) * a.other + c.aux < a.bign;
          const C2<T> y = cmul(v[r], cj ? w[r - s] : conjc(w[r - s]));
          v[r] = on ? y : C2<T>{T(0), T(0)};
        }
      }
    } else if ((op == OP_C2C || op == OP_PASSA) && a.rot_in) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = gload(c.in + rot_index(at(r), a.rot_in, a.nin) * es);
    } else {
      const T *p = c.in + j * es;
      const auto step = NR * es;
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = gload(CLAMP ? c.in + at(r) * es : p + r * step);
    }
  } else if (op == OP_BLUE) {
    const int n = int(a.bign);
#pragma unroll
    for (int s = 0; s < R; s += S) {
      C2<T> w[S];
#pragma unroll
      for (int r = s; r < R && r < s + S; ++r) {  // element (j + rot_in) mod n, times the chirp at j
        const int jj = at(r) < n ? at(r) : 0;
        w[r - s] = a.t0[jj];
        v[r] = gload(c.in + rot_index(jj, a.rot_in, n) * es);
      }
#pragma unroll
      for (int r = s; r < R && r < s + S; ++r) {
        const C2<T> y = cmul(v[r], cj ? w[r - s] : conjc(w[r - s]));
        v[r] = at(r) < n ? y : C2<T>{T(0), T(0)};
      }
    }
  } else if (op == OP_R2C_EVEN) {
    const T *p = c.in + 2 * j * es;
    const auto step = 2 * NR * es;
    if (FLAT || es == 1) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = gload(CLAMP ? c.in + 2 * at(r) * es : p + r * step);
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const T *q = CLAMP ? c.in + 2 * at(r) * es : p + r * step;
        v[r] = C2<T>{q[0], q[es]};
      }
    }
  } else if (op == OP_R2C_ODD) {
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = C2<T>{c.in[at(r) * es], T(0)};
  } else if (op == OP_C2R_EVEN) {
    const int h = a.f.n;
    const T *p = c.in + j * es, *pm = c.in + (h - j) * es;
    const auto step = NR * es;
    C2<T> xm[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      v[r] = gload(CLAMP ? c.in + at(r) * es : p + r * step);
      xm[r] = gload(CLAMP ? c.in + (h - at(r)) * es : pm - r * step);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      C2<T> x = v[r], y = xm[r];
      const int jj = at(r);
      if (!cj) y.y = -y.y;  // conj of the mirrored bin (of the conjugated input)
      else x.y = -x.y;
      if (jj == 0) x.y = y.y = T(0);
      const C2<T> A = x + y;
      const C2<T> B = cmul(x - y, conjc(a.t0[jj]));
      v[r] = C2<T>{A.x - B.y, A.y + B.x};
    }
  } else {  // OP_C2R_ODD: bin j, or the conjugate of bin n - j
    const int n = a.f.n;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int jj = at(r);
      v[r] = gload(c.in + (2 * jj < n ? jj : n - jj) * es);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int jj = at(r);
      if ((2 * jj < n) == cj) v[r].y = -v[r].y;
      if (jj == 0) v[r].y = T(0);
    }
  }
  if (op != OP_BLUE && op != OP_BLUEROW && op != OP_R2C_EVEN && op != OP_R2C_ODD) {
    if (a.dir > T(0)) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = C2<T>{v[r].y, v[r].x};
    }
  }
}

// Bins j + r ns (r < R), with the op's post-processing.  CLAMP: those beyond
// the line are left out.  FLAT: 24-bit strides.
template <typename T, int OP, int R, bool CLAMP = false, bool FLAT = false>
__device__ __forceinline__ void op_store(const LineArgs<T> &a, const MixCtx<T> &c, int j, int ns,
                                         C2<T> *v) {
  constexpr int S = kFactors<T, OP, R>;
  const bool cj = (a.sub & SUB_CONJ) != 0;
  using Es = std::conditional_t<FLAT, Stride24, int64_t>;
  const Es es = Es(a.eso);
  const int op = op_of<OP>(a);
  auto in_line = [&](int r) { return !CLAMP || j + r * ns < a.f.n; };
  if (is_blue(op) || (op != OP_R2C_ODD && a.dir > T(0))) {  // the inverse transform ran on exchanged parts
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = C2<T>{v[r].y, v[r].x};
  }
  T *p = c.out + j * es;
  const auto step = ns * es;
  if (op == OP_C2C || op == OP_PASSB) {
    if (a.rot_out) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (in_line(r))
          gstore(c.out + rot_index(j + r * ns, a.rot_out, a.nout) * es, a.fct * v[r]);
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (in_line(r)) gstore(p + r * step, a.fct * v[r]);
    }
  } else if (op == OP_PASSA) {
    // a slice's factors first, without a condition around their loads
    if (a.sub & SUB_FINAL) {  // Bluestein columns, last pass: chirp and fct, m < n
#pragma unroll
      for (int s = 0; s < R; s += S) {
        C2<T> w[S];
#pragma unroll
        for (int r = s; r < R && r < s + S; ++r) {
          const int64_t m = c.aux + int64_t(j + r * ns) * a.other;
          w[r - s] = a.t0[m < a.bign ? m : c.aux];
        }
#pragma unroll
        for (int r = s; r < R && r < s + S; ++r) {
          const int k = j + r * ns;
          const int64_t m = c.aux + int64_t(k) * a.other;
          if (in_line(r) && m < a.bign)
            gstore(c.out + blue_col_offset(k, m, a.rot_out, a.bign, c.aux, es, a.other),
                   a.fct * cmul(v[r], cj ? w[r - s] : conjc(w[r - s])));
        }
      }
    } else {
#pragma unroll
      for (int s = 0; s < R; s += S) {
        C2<T> w[S];
#pragma unroll
        for (int r = s; r < R && r < s + S; ++r)
          w[r - s] = step_twiddle(a, CLAMP ? min(j + r * ns, a.f.n - 1) : j + r * ns, c.aux);
#pragma unroll
        for (int r = s; r < R && r < s + S; ++r)
          if (in_line(r)) gstore(p + r * step, cmul(v[r], dirw(w[r - s], a.dir)));
      }
    }
  } else if (op == OP_BLUEROW) {
#pragma unroll
    for (int s = 0; s < R; s += S) {
      C2<T> w[S];
#pragma unroll
      for (int r = s; r < R && r < s + S; ++r)
        w[r - s] = step_twiddle(a, CLAMP ? min(j + r * ns, a.f.n - 1) : j + r * ns, c.aux);
#pragma unroll
      for (int r = s; r < R && r < s + S; ++r)
        if (in_line(r)) gstore(p + r * step, cmul(v[r], conjc(w[r - s])));
    }
  } else if (op == OP_BLUE) {  // bin k < n, chirped, to (k + rot_out) mod n
#pragma unroll
    for (int s = 0; s < R; s += S) {
      C2<T> w[S];
#pragma unroll
      for (int r = s; r < R && r < s + S; ++r)
        w[r - s] = a.t0[j + r * ns < a.nout ? j + r * ns : 0];
#pragma unroll
      for (int r = s; r < R && r < s + S; ++r) {
        const int k = j + r * ns;
        if (in_line(r) && k < a.nout)
          gstore(c.out + rot_index(k, a.rot_out, a.nout) * es,
                 a.fct * cmul(v[r], cj ? w[r - s] : conjc(w[r - s])));
      }
    }
  } else if (op == OP_R2C_ODD) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (in_line(r) && j + r * ns < a.nout) {
        if (cj) v[r].y = -v[r].y;
        gstore(p + r * step, a.fct * v[r]);
      }
  } else if (op == OP_C2R_EVEN) {
    T *q = c.out + 2 * j * es;
    if (FLAT || es == 1) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (in_line(r)) gstore(q + 2 * r * step, a.fct * v[r]);
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (in_line(r)) {
          q[2 * r * step] = a.fct * v[r].x;
          q[2 * r * step + es] = a.fct * v[r].y;
        }
    }
  } else if (op == OP_C2R_ODD) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (in_line(r)) p[r * step] = a.fct * v[r].x;
  }
}

// Bluestein kernel product on bins j + r ns, leaving the parts exchanged for
// the inverse transform.
template <typename T, int OP, int R>
__device__ __forceinline__ void kernel_product(const LineArgs<T> &a, const MixCtx<T> &c, int j,
                                               int ns, C2<T> *v) {
  const T cs = (a.sub & SUB_CONJ) != 0 ? T(-1) : T(1);
  const bool row = op_of<OP>(a) == OP_BLUEROW;
  const C2<T> *kp = row ? a.t2 + int64_t(c.aux) * a.f.n : a.t1;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    C2<T> w = kp[j + r * ns];
    w.y *= cs;
    const C2<T> y = cmul(v[r], w);
    v[r] = C2<T>{y.y, y.x};
  }
}

// Bin k of a real line from bins k and h - k of its half-length spectrum.
template <typename T>
__device__ __forceinline__ void real_bin(const LineArgs<T> &a, int k, int h, C2<T> zk, C2<T> zm,
                                         T *to) {
  C2<T> X;
  if (k == 0 || k == h) {
    X = C2<T>{k == 0 ? zk.x + zk.y : zk.x - zk.y, T(0)};
  } else {
    zm = conjc(zm);
    const C2<T> fe = T(0.5) * (zk + zm);
    const C2<T> dd = zk - zm;
    X = fe + cmul(a.t0[k], C2<T>{T(0.5) * dd.y, T(-0.5) * dd.x});
  }
  if ((a.sub & SUB_CONJ) != 0) X.y = -X.y;
  gstore(to, a.fct * X);
}

// One forward stage of radix R (first: inputs from global memory; last:
// outputs to global memory, or for Bluestein on through the kernel product
// into the first backward stage).
template <typename T, int OP, int R, int FORM = 0>
__device__ __forceinline__ void mix_stage(const LineArgs<T> &a, const MixGeom &m,
                                          const MixStage &st, const MixCtx<T> &c, bool first,
                                          bool last) {
  constexpr int QM = !(FORM & kShort) && kMaxElems<T> / R > 0 ? kMaxElems<T> / R : 1;
  const int op = op_of<OP>(a);
  const int NR = FORM & kShort ? 1 : st.nr, ns = FORM & kShort ? 1 : st.ns;
  constexpr bool FLAT = (FORM & kFlat) != 0;
  const bool from_lds = !first || OP == OP_R2R || OP == OP_ANY || FLAT;
  const C2<T> *tw = a.tw + st.twoff;
  C2<T> v[QM][R];
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int j = c.j + q * m.T;
    if ((FORM & kShort || q < st.q) && c.ok && j < NR) {
      bool loaded = false;
      if constexpr (OP != OP_ANY && OP != OP_R2R)
        if (!from_lds) {
          op_load<T, OP, R>(a, c, j, NR, v[q]);
          loaded = true;
        }
      if (!loaded) {
        const int b = FORM & kShort ? 0 : fdiv(j, ns, st.invns), k = j - b * ns;
        const C2<T> *s = c.ln + b * st.pbi + k;
        const int rs = FORM & kShort ? 1 : st.rs;
#pragma unroll
        for (int r = 0; r < R; ++r) v[q][r] = s[r * rs];
        if (!first) {
#pragma unroll
          for (int r = 1; r < R; ++r) v[q][r] = cmul(v[q][r], tw[(r - 1) * ns + k]);
        }
      }
      bfly<R>(v[q]);
    }
  }
  if constexpr (FORM == kShort && OP == OP_R2C_EVEN) {  // the whole spectrum is in v
    if (c.ok) {
#pragma unroll
      for (int k = 0; k <= R; ++k)
        real_bin(a, k, R, v[0][k % R], v[0][(R - k) % R], c.out + k * a.eso);
    }
    return;
  }
  if constexpr (OP != OP_ANY) {
    if (elem_store(op) && !is_blue(op) && last && !FLAT) {
#pragma unroll
      for (int q = 0; q < QM; ++q) {
        const int j = c.j + q * m.T;
        if ((FORM & kShort || q < st.q) && c.ok && j < NR)
          op_store<T, OP, R>(a, c, j, ns, v[q]);
      }
      return;
    }
  }
  if (is_blue(op)) {
    if (last) {  // ns == NR: k == j
#pragma unroll
      for (int q = 0; q < QM; ++q) {
        const int j = c.j + q * m.T;
        if (q < st.q && c.ok && j < NR) {
          kernel_product<T, OP, R>(a, c, j, ns, v[q]);
          bfly<R>(v[q]);
          if (!first) {
#pragma unroll
            for (int r = 1; r < R; ++r) v[q][r] = cmul(v[q][r], tw[(r - 1) * ns + j]);
          } else if constexpr (OP != OP_ANY) {
            op_store<T, OP, R>(a, c, j, NR, v[q]);
          }
        }
      }
      if (first && OP != OP_ANY) return;
      __syncthreads();
#pragma unroll
      for (int q = 0; q < QM; ++q) {
        const int j = c.j + q * m.T;
        if (q < st.q && c.ok && j < NR) {
          C2<T> *d = c.ln + j;
#pragma unroll
          for (int r = 0; r < R; ++r) d[r * st.rs] = v[q][r];
        }
      }
      __syncthreads();
      return;
    }
  }
  if (from_lds) __syncthreads();
  const bool sw = last && OP == OP_R2R && a.dir > T(0);  // read back in its own order
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int j = c.j + q * m.T;
    if ((FORM & kShort || q < st.q) && c.ok && j < NR) {
      const int b = FORM & kShort ? 0 : fdiv(j, ns, st.invns), k = j - b * ns;
      C2<T> *d = c.ln + b * st.pbo + k;
#pragma unroll
      for (int r = 0; r < R; ++r) d[r * ns] = swapri(v[q][r], sw);
    }
  }
  __syncthreads();
}

// One stage of the Bluestein inverse transform, undone backwards: reads where
// the forward stage wrote, butterfly, twiddles, writes where it read (the
// first stage: to global memory).
template <typename T, int OP, int R>
__device__ __forceinline__ void mix_unstage(const LineArgs<T> &a, const MixGeom &m,
                                            const MixStage &st, const MixCtx<T> &c, bool first) {
  constexpr int QM = kMaxElems<T> / R > 0 ? kMaxElems<T> / R : 1;
  const int NR = st.nr, ns = st.ns;
  const C2<T> *tw = a.tw + st.twoff;
  C2<T> v[QM][R];
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int j = c.j + q * m.T;
    if (q < st.q && c.ok && j < NR) {
      const int b = fdiv(j, ns, st.invns), k = j - b * ns;
      const C2<T> *d = c.ln + b * st.pbo + k;
#pragma unroll
      for (int r = 0; r < R; ++r) v[q][r] = d[r * ns];
      bfly<R>(v[q]);
      if (!first) {
#pragma unroll
        for (int r = 1; r < R; ++r) v[q][r] = cmul(v[q][r], tw[(r - 1) * ns + k]);
      } else if constexpr (OP != OP_ANY) {
        op_store<T, OP, R>(a, c, j, NR, v[q]);
      }
    }
  }
  if (first && OP != OP_ANY) return;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int j = c.j + q * m.T;
    if (q < st.q && c.ok && j < NR) {
      const int b = fdiv(j, ns, st.invns), k = j - b * ns;
      C2<T> *s = c.ln + b * st.pbi + k;
#pragma unroll
      for (int r = 0; r < R; ++r) s[r * st.rs] = v[q][r];
    }
  }
  __syncthreads();
}

// Real-to-real modes: f(mode) with the mode a compile-time constant for the
// DCT / DST types, so that the elements of a batch are in one stretch of code
// and their loads in flight together.
template <typename F>
__device__ __forceinline__ void with_pre_mode(int mode, F &&f) {
  switch (mode) {
#define RFH_MODE(M) \
  case M: f(std::integral_constant<int, M>{}); break;
    RFH_MODE(kPreDct1) RFH_MODE(kPreDst1) RFH_MODE(kPreType4) RFH_MODE(kPreDct2N)
    RFH_MODE(kPreDst2N) RFH_MODE(kPreDct3N) RFH_MODE(kPreDst3N)
    default: f(mode);
  }
}
template <typename F>
__device__ __forceinline__ void with_post_mode(int mode, F &&f) {
  switch (mode) {
    RFH_MODE(kPostDct1) RFH_MODE(kPostDst1) RFH_MODE(kPostDct4) RFH_MODE(kPostDst4)
    RFH_MODE(kPostDct2N) RFH_MODE(kPostDst2N) RFH_MODE(kPostDct3N) RFH_MODE(kPostDst3N)
#undef RFH_MODE
    default: f(mode);
  }
}

// The whole line to LDS, in order, a batch of loads of a thread in flight.
constexpr int kLineBatch = 8;
template <typename T, int OP, int FORM>
__device__ __forceinline__ void load_line(const LineArgs<T> &a, const MixGeom &m,
                                          const MixCtx<T> &c) {
  constexpr bool FLAT = (FORM & kFlat) != 0;
  const Walk<T, FORM> w(m, c, a.f.n);
  // (short lines leave most of a large batch empty; two loads an element)
  constexpr int B = FLAT && ((FORM & kShort) || OP == OP_C2R_EVEN) ? 4 : kLineBatch;
  auto walk = [&](auto &&load) {
    for (int e = w.first; e < w.total; e += B * w.step) {
      C2<T> v[B], *to[B];
#pragma unroll
      for (int r = 0; r < B; ++r) {
        MixCtx<T> at;
        const int p = w.place(min(e + r * w.step, w.total - 1), at);
        to[r] = at.ln + p;
        load(at, p, &v[r]);
      }
#pragma unroll
      for (int r = 0; r < B; ++r)
        if (e + r * w.step < w.total) *to[r] = v[r];
    }
  };
  if (w.on) {
    if constexpr (OP == OP_R2R) {
      with_pre_mode(a.sub & 0xff, [&](auto mode) {
        walk([&](const MixCtx<T> &at, int p, C2<T> *v) {
          *v = swapri(pre_elem<T, int>(mode, at.in, FLAT ? 1 : a.esi, int(a.bign), a.f.n, p,
                                       (a.sub & R2R_ORTHO) != 0, (a.sub & R2R_CONJ) != 0,
                                       (a.sub & R2R_FLIP) != 0, root_of<(FORM & kSinCos) != 0>(a)),
                      a.dir > T(0));
        });
      });
    } else if constexpr (OP == OP_ANY) {
      for (int e = c.j; e < a.f.n; e += B * w.step) {
        C2<T> v[B];
        op_load<T, OP, B, true>(a, c, e, w.step, v);
#pragma unroll
        for (int r = 0; r < B; ++r)
          if (e + r * w.step < a.f.n) c.ln[e + r * w.step] = v[r];
      }
    } else if constexpr (FLAT) {
      walk([&](const MixCtx<T> &at, int p, C2<T> *v) { op_load<T, OP, 1, false, true>(a, at, p, 0, v); });
    } else {
      for (int e = c.j; e < a.f.n; e += w.step) {
        C2<T> v;
        op_load<T, OP, 1>(a, c, e, 0, &v);
        c.ln[e] = v;
      }
    }
  }
  __syncthreads();
}

// ... and from LDS.
template <typename T, int OP, int FORM>
__device__ __forceinline__ void store_line(const LineArgs<T> &a, const MixGeom &m,
                                           const MixCtx<T> &c) {
  const int count = OP == OP_R2C_ODD ? a.nout : a.f.n;
  const Walk<T, FORM> w(m, c, count);
  if (!w.on) return;
  if constexpr (OP == OP_ANY) {
    for (int e = c.j; e < a.f.n; e += kLineBatch * w.step) {
      C2<T> v[kLineBatch];
#pragma unroll
      for (int r = 0; r < kLineBatch; ++r) v[r] = c.ln[min(e + r * w.step, a.f.n - 1)];
      op_store<T, OP, kLineBatch, true>(a, c, e, w.step, v);
    }
  } else {
    constexpr int B = 4;
    for (int e = w.first; e < w.total; e += B * w.step) {
      MixCtx<T> at[B];
      C2<T> v[B];
      int p[B];
#pragma unroll
      for (int r = 0; r < B; ++r) {
        p[r] = w.place(min(e + r * w.step, w.total - 1), at[r]);
        v[r] = at[r].ln[p[r]];
      }
#pragma unroll
      for (int r = 0; r < B; ++r)
        if (e + r * w.step < w.total)
          op_store<T, OP, 1, false, (FORM & kFlat) != 0>(a, at[r], p[r], 0, &v[r]);
    }
  }
}

// Inputs mm and R - mm of a prime stage's butterfly, twiddled, into the sums of
// output pairs k0 .. k0 + q - 1 (q <= Q).
template <typename T, int Q, int PM>
__device__ __forceinline__ void prime_step(const MixStage &st, const C2<T> *s, const C2<T> *tw,
                                           int k, const C2<T> *g, int k0, int mm, C2<T> &sum,
                                           C2<T> (&A)[PM], C2<T> (&B)[PM], int (&idx)[PM]) {
  const int R = st.radix, ns = st.ns;
  C2<T> xp = s[mm * st.rs], xm = s[(R - mm) * st.rs];
  if (ns > 1) {
    xp = cmul(xp, tw[(mm - 1) * ns + k]);
    xm = cmul(xm, tw[(R - mm - 1) * ns + k]);
  }
  const C2<T> t = xp + xm, d = xp - xm;
  sum = sum + t;
#pragma unroll
  for (int p = 0; p < Q; ++p) {
    if (Q == 1 || p < st.q) {
      idx[p] += k0 + p;
      if (idx[p] >= R) idx[p] -= R;
      const C2<T> w = g[idx[p]];
      A[p] = A[p] + w.x * t;
      B[p] = B[p] + w.y * d;
    }
  }
}
template <typename T, int Q, int PM>
__device__ __forceinline__ void prime_sums(const MixStage &st, const C2<T> *s, const C2<T> *tw,
                                           int k, const C2<T> *g, int k0, C2<T> &sum,
                                           C2<T> (&A)[PM], C2<T> (&B)[PM], int (&idx)[PM]) {
  const int H = (st.radix - 1) / 2;
  int mm = 1;
  if constexpr (Q <= 3) {  // few lines: a chain of loads, some iterations' in flight
    constexpr int U = Q == 1 ? 4 : 2;
    for (; mm + U - 1 <= H; mm += U) {
#pragma unroll
      for (int u = 0; u < U; ++u) prime_step<T, Q, PM>(st, s, tw, k, g, k0, mm + u, sum, A, B, idx);
    }
  }
  for (; mm <= H; ++mm) prime_step<T, Q, PM>(st, s, tw, k, g, k0, mm, sum, A, B, idx);
}

// A stage of a prime radix R above 17: st.q output pairs (kk, R - kk) of one
// butterfly per thread, accumulated over the symmetric sums of its inputs,
// which are read (and twiddled) once for all of them.  Unit u = chunk NR +
// butterfly, so lanes share a chunk and the roots come from LDS as broadcasts.
template <typename T, int OP, int FORM>
__device__ __forceinline__ void mix_prime_stage(const LineArgs<T> &a, const MixGeom &m,
                                                const MixStage &st, const MixCtx<T> &c,
                                                const C2<T> *roots, bool first, bool last) {
  constexpr bool FEW = !(FORM & kPrime) && OP != OP_ANY;
  constexpr int PM = FEW ? kFewPairs : kMaxElems<T> / 2;
  const int R = st.radix, NR = st.nr, ns = st.ns, H = (R - 1) / 2;
  const C2<T> *tw = a.tw + st.twoff;
  constexpr bool FLAT = (FORM & kFlat) != 0;
  if (first && OP != OP_R2R && OP != OP_ANY && !FLAT) load_line<T, OP, FORM>(a, m, c);  // an input serves several threads
  const int ch = fdiv(c.j, NR, 1.0f / float(NR)), j = c.j - ch * NR;
  const int k0 = ch * st.q;  // first pair of the chunk
  const bool on = c.ok && k0 <= H;
  const int b = fdiv(j, ns, st.invns), k = j - b * ns;
  const C2<T> *s = c.ln + b * st.pbi + k;
  const C2<T> *g = roots + st.genoff;
  C2<T> x0{T(0), T(0)}, sum{T(0), T(0)}, A[PM], B[PM];
  if (on) {
    x0 = sum = s[0];
    int idx[PM];
#pragma unroll
    for (int p = 0; p < PM; ++p) {
      A[p] = x0;
      B[p] = C2<T>{T(0), T(0)};
      idx[p] = 0;
    }
    if (FEW && st.q == 1) prime_sums<T, 1, PM>(st, s, tw, k, g, k0, sum, A, B, idx);
    else prime_sums<T, PM, PM>(st, s, tw, k, g, k0, sum, A, B, idx);
  }
  // outputs: bin kk and bin R - kk of the butterfly
  const bool lds = OP == OP_ANY || !(elem_store(op_of<OP>(a)) && last && !FLAT);
  const bool sw = lds && last && OP == OP_R2R && a.dir > T(0);
  if (lds) __syncthreads();
  if (on) {
#pragma unroll
    for (int p = 0; p < PM; ++p) {
      const int kk = k0 + p;
      if (p < st.q && kk <= H) {
        C2<T> lo = {A[p].x + B[p].y, A[p].y - B[p].x}, hi = {A[p].x - B[p].y, A[p].y + B[p].x};
        if (kk == 0) lo = sum;
        if (lds) {
          C2<T> *d = c.ln + b * st.pbo + k;
          d[kk * ns] = swapri(lo, sw);
          if (kk) d[(R - kk) * ns] = swapri(hi, sw);
        } else if constexpr (OP != OP_ANY) {  // last stage: ns == NR, bins j + kk ns
          op_store<T, OP, 1>(a, c, j + kk * ns, 0, &lo);
          if (kk) op_store<T, OP, 1>(a, c, j + (R - kk) * ns, 0, &hi);
        }
      }
    }
  }
  if (lds) __syncthreads();
}

#define RFH_SHORT_RADICES(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9)
#define RFH_MIX_RADICES(X) \
  X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16) X(17)

// The place of thread t in its group: the line it works on and its index in
// it.  Contiguous lines: a line's threads are adjacent (runs along the line);
// interleaved lines: adjacent threads take the same place of adjacent lines.
// SHORT: a thread a line.
template <typename T, bool SHORT>
__device__ __forceinline__ MixCtx<T> mix_place(const LineArgs<T> &a, const MixGeom &m,
                                               int64_t tile, C2<T> *lds, bool lfast) {
  const int t = threadIdx.x;
  int l = t, j = 0;
  if (SHORT) {
  } else if (lfast) {
    l = t & (m.L - 1);
    j = t >> m.log2L;
  } else {
    l = m.L == 1 ? 0 : fdiv(t, m.T, m.invT);
    j = t - l * m.T;
  }
  MixCtx<T> c;
  const int64_t b = tile * m.L + l;
  c.line = l < m.L && b < a.nlines;
  c.ok = c.line && (SHORT || j < m.T);
  const LineOffsets o = c.line ? line_offsets(b, a.nb, a.bdim, a.bsi, a.bso, a.auxdim)
                             : LineOffsets{0, 0, 0};
  c.in = a.in + o.oi;
  c.out = a.out + o.oo;
  c.aux = o.aux;
  c.j = j;
  c.ln = lds + (c.line ? l : 0) * m.ld;
  c.in0 = a.in + (a.nb ? tile * m.L * a.bsi[0] : 0);
  c.out0 = a.out + (a.nb ? tile * m.L * a.bso[0] : 0);
  c.nl = int(min(int64_t(m.L), a.nlines - tile * m.L));
  c.lds = lds;
  return c;
}

// One tile (m.L lines from line tile m.L on) of a line set.  Ends without a
// barrier: a caller that runs several tiles puts one between them.
template <typename T, int OP, int FORM = 0>
__device__ __forceinline__ void mix_body(const LineArgs<T> &a, const MixGeom &m, int64_t tile,
                                         unsigned char *smem) {
  const int op = op_of<OP>(a);
  C2<T> *lds = reinterpret_cast<C2<T> *>(smem);
  MixCtx<T> c = mix_place<T, (FORM & kShort) != 0>(a, m, tile, lds, a.lfast_in != 0);
  C2<T> *roots = lds + m.L * m.ld;
  if (!(FORM & kShort) && m.ngen) {
    for (int i = threadIdx.x; i < m.ngen; i += blockDim.x) roots[i] = a.gen[i];
    __syncthreads();
  }
  if (m.nst == 0) {  // lines of one element
    if (c.ok && c.j == 0) {
      C2<T> v[1];
      if constexpr (OP == OP_R2R)
        v[0] = pre_elem<T, int>(a.sub & 0xff, c.in, a.esi, int(a.bign), a.f.n, 0,
                                (a.sub & R2R_ORTHO) != 0, (a.sub & R2R_CONJ) != 0,
                                (a.sub & R2R_FLIP) != 0, root_of<(FORM & kSinCos) != 0>(a));
      else
        op_load<T, OP, 1>(a, c, 0, 0, v);
      if (is_blue(op)) kernel_product<T, OP, 1>(a, c, 0, 0, v);
      if (elem_store(op)) op_store<T, OP, 1>(a, c, 0, 0, v);
      else c.ln[0] = v[0];
    }
    __syncthreads();
  }
  // the real-to-real modes' heavier loads stay out of the unrolled stages
  constexpr bool FLAT = (FORM & kFlat) != 0;
  if ((OP == OP_R2R || OP == OP_ANY || FLAT) && m.nst) load_line<T, OP, FORM>(a, m, c);
#define RFH_CASE(R) \
  case R: mix_stage<T, OP, R, FORM>(a, m, st, c, first, last); break;
  if constexpr (FORM & kShort) {
    const MixStage &st = m.st[0];
    constexpr bool first = true, last = true;
    if (m.nst) {
      switch (st.radix) {
        RFH_SHORT_RADICES(RFH_CASE)
        default: break;
      }
    }
  }
  for (int s = 0; !(FORM & kShort) && s < m.nst; ++s) {
    const MixStage &st = m.st[s];
    const bool first = s == 0, last = s == m.nst - 1;
    switch (st.radix) {
      RFH_MIX_RADICES(RFH_CASE)
#undef RFH_CASE
      default:
        if constexpr (!is_blue_op(OP) && !(FORM == kFlat))
          mix_prime_stage<T, OP, FORM>(a, m, st, c, roots, first, last);
        break;
    }
    // from the first exchange on, threads take the places of the output side
    if (first && !last && a.lfast_out != a.lfast_in)
      c = mix_place<T, false>(a, m, tile, lds, a.lfast_out != 0);
  }
  if (is_blue(op)) {
    for (int s = m.nst - 2; s >= 0; --s) {
      const MixStage &st = m.st[s];
      switch (st.radix) {
#define RFH_CASE(R) \
  case R: mix_unstage<T, OP, R>(a, m, st, c, s == 0); break;
        RFH_MIX_RADICES(RFH_CASE)
#undef RFH_CASE
        default: break;
      }
    }
  }
  if constexpr (OP == OP_ANY || FLAT)  // the bins are in LDS, in order
    if (m.nst && elem_store(op)) store_line<T, OP, FORM>(a, m, c);
  // bins k and h - k of the half-length spectrum (FORM == kShort: stored already)
  if (op == OP_R2C_EVEN && !(FORM == kShort && m.nst)) {
    const int h = a.f.n;
    const Walk<T, FORM> w(m, c, h + 1);
    if (w.on) {
      for (int e = w.first; e < w.total; e += w.step) {
        MixCtx<T> at;
        const int k = w.place(e, at);
        const bool end = k == 0 || k == h;
        real_bin(a, k, h, at.ln[end ? 0 : k], at.ln[end ? 0 : h - k],
                 at.out + (FLAT ? k * Stride24(a.eso) : k * a.eso));
      }
    }
  }
  if constexpr (OP == OP_R2R) {
    const Walk<T, FORM> w(m, c, a.nout);
    if (w.on) {
      with_post_mode((a.sub >> 8) & 0xff, [&](auto mode) {
        for (int e = w.first; e < w.total; e += kLineBatch * w.step) {
          T y[kLineBatch], *to[kLineBatch];
#pragma unroll
          for (int r = 0; r < kLineBatch; ++r) {
            MixCtx<T> at;
            const int k = w.place(min(e + r * w.step, w.total - 1), at);
            const C2<T> *ln = at.ln;
            y[r] = a.fct * post_elem<T, int>(mode, [&](int q) { return ln[q]; }, int(a.bign), k,
                                             (a.sub & R2R_ORTHO) != 0, (a.sub & R2R_FLIP) != 0,
                                             root_of<(FORM & kSinCos) != 0>(a));
            to[r] = at.out + (FLAT ? k : k * a.eso);
          }
#pragma unroll
          for (int r = 0; r < kLineBatch; ++r)
            if (e + r * w.step < w.total) *to[r] = y[r];
        }
      });
    }
  }
}

}  // namespace dev
}  // namespace rfh
