// mixgeom.hpp -- the general line kernel's (mixline.hpp) radices, threads and
// LDS layout for a line length.  Plain C++, unit-tested on the host.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace rfh {

// Elements a thread may hold per stage and threads of the largest workgroup:
// bounded by the registers of 1024 threads (complex64: 128 each) or 768
// (complex128: 168 each).
constexpr int mix_max_elems(bool dbl) { return dbl ? 18 : 20; }
constexpr int mix_max_threads(bool dbl) { return dbl ? 768 : 1024; }
constexpr int kMixLines = 256;  // lines per group, at most
// one wave on every SIMD (256 CUs of four)
constexpr int64_t kFillThreads = 256 * 4 * 64;

// A launch's threads are counted in 31 bits: line sets of more groups run in
// several launches.  f(first group, groups) for each.
constexpr int64_t kLaunchThreads = 0x7fffffff;
template <typename F>
void for_launches(int64_t groups, int threads, F &&f) {
  const int64_t most = kLaunchThreads / threads;
  for (int64_t g = 0; g < groups; g += most) f(g, std::min(most, groups - g));
}

constexpr int kMixStages = 10;

struct MixStage {
  int radix;   // 2 .. 17, or a larger odd prime
  int q;       // butterflies per thread (larger primes: output pairs per thread)
  int nr;      // N / radix
  int ns;      // product of the earlier radices
  int rs;      // LDS distance of a butterfly's inputs
  int pbi;     // LDS pitch of a block of ns elements (input layout)
  int pbo;     // LDS pitch of a block of ns radix elements (output layout)
  int twoff;   // twiddles W_{ns radix}^{k r} at tw + twoff + (r - 1) ns + k
  int genoff;  // larger primes: roots (cos, sin)(2 pi q / radix)
  float invns;
};

struct MixGeom {
  int T;      // threads per line
  int L;      // lines per group
  int log2L;  // interleaved lines: L is a power of two
  int nst;
  int ld;     // LDS elements per line
  int ngen;   // roots of larger primes copied to LDS behind the lines
  int flat;   // the group's lines are loaded and stored one after another
  int flat_in, flat_out;  // ... and lie this many scalars apart
  float invT;
  MixStage st[kMixStages];
};

// Lines of at most one butterfly of a radix up to 9, a thread each.
inline bool short_lines(const MixGeom &m) {
  return m.nst == 0 || (m.nst == 1 && m.st[0].radix <= 9 && m.st[0].q == 1);
}

// Whether a thread takes at most kFewPairs of the output pairs of a butterfly of
// a prime above 17: sums in a form of the kernel of their own, without the
// branches and registers of more pairs, a lone pair's loads several iterations
// ahead.  us, before the general kernel was rewritten / since / now: 24 lines of
// 122 complex64 11.6 / 16.6 / 10.9, of 194 complex128 15.0 / 24.8 / 13.6.
constexpr int kFewPairs = 3;
inline bool few_pairs(const MixGeom &m) {
  for (int s = 0; s < m.nst; ++s)
    if (m.st[s].radix > 17 && m.st[s].q > kFewPairs) return false;
  return true;
}

// Threads a line of n needs when each may hold 16 elements of a stage's
// butterflies, and how evenly the stages use them: the sum over the stages of
// (elements held by all threads, idle places included) / n; among equals the
// smaller radices, which a small launch can spread over more threads.
inline double radix_waste(uint64_t n, const std::vector<int> &r) {
  uint64_t t = 1;
  for (int R : r) t = std::max<uint64_t>(t, (n / R + (R > 16 ? 1 : 16 / R) - 1) / (R > 16 ? 1 : 16 / R));
  double w = 0;
  for (int R : r) w += double((n / R + t - 1) / t * R * t) / double(n) + 1e-3 * R;
  return w;
}

// All products of n as `left` radices <= `top` in descending order; keeps the
// one whose stages waste the fewest places.
inline void radix_search(uint64_t n, uint64_t rest, int left, int top, std::vector<int> &cur,
                         std::vector<int> &best, double &best_w) {
  if (left == 0) {
    if (rest != 1) return;
    const double w = radix_waste(n, cur);
    if (best.empty() || w < best_w) {
      best = cur;
      best_w = w;
    }
    return;
  }
  uint64_t most = 1;
  for (int i = 0; i < left; ++i) most *= uint64_t(top);
  if (rest > most) return;
  for (int R = top; R >= 2; --R) {
    if (rest % R) continue;
    cur.push_back(R);
    radix_search(n, rest / R, left - 1, R, cur, best, best_w);
    cur.pop_back();
  }
}

// The fewest radices of 2 .. 17 (each stage is an exchange through LDS), among
// those the ones whose butterflies fill a line's threads best (1000 = 10 x 10 x
// 10, 1920 = 16 x 15 x 8), the largest first (the first stage has no
// twiddles); then the primes above 17.
inline std::vector<int> even_radices(uint64_t n) {
  std::vector<int> r;
  uint64_t smooth = 1, rest = n;
  for (uint64_t d : {2, 3, 5, 7, 11, 13, 17})
    while (rest > 1 && rest % d == 0) {
      rest /= d;
      smooth *= d;
    }
  double w = 0;
  if (smooth > 1)
    for (int count = 1; r.empty(); ++count) {
      std::vector<int> cur;
      radix_search(smooth, smooth, count, 17, cur, r, w);
    }
  for (uint64_t d = 19; d * d <= rest; d += 2)
    while (rest % d == 0) {
      r.push_back(int(d));
      rest /= d;
    }
  if (rest > 1) r.push_back(int(rest));
  return r;
}

// Powers of two: radix 16 first, then 8 / 4 / 2, the schedule the specialised
// kernels are compiled for.
inline std::vector<int> mix_radices(uint64_t n) {
  if (n < 2 || (n & (n - 1)) != 0) return even_radices(n);
  std::vector<int> r;
  for (; n >= 16; n /= 16) r.push_back(16);
  if (n > 1) r.push_back(int(n));
  return r;
}

// LDS pitch of the blocks of nb elements a stage writes in runs of ns: the
// least padding that spreads the 64 lanes' writes over the banks (a pass of
// the LDS takes 32 lanes of 8 bytes or 16 of 16 bytes).
inline int block_pitch(int nb, int ns, bool dbl) {
  const int G = dbl ? 16 : 32;
  if (ns >= G) return nb;
  int best = nb, best_c = 1 << 30;
  for (int P = nb; P <= nb + 8; ++P) {
    int c = 0;
    for (int g = 0; g < 64; g += G) {
      int hit[32] = {}, most = 0;
      for (int i = g; i < g + G; ++i) most = std::max(most, ++hit[(i / ns * P + i % ns) % G]);
      c += most;
    }
    if (c < best_c) {
      best_c = c;
      best = P;
    }
  }
  return best;
}

// Geometry for lines of desc (n, nst, st[] with radix, ns, twoff, genoff; pbo[s]
// the pitch of stage s's blocks).  `want`: adjacent lines an interleaved group
// should hold (0: 128-byte row segments).  L == 0: a line does not fit.
template <typename Desc>
MixGeom mix_geometry(const Desc &f, const int *pbo, bool dbl, int64_t nlines, bool inter, int want,
                     size_t lds_bytes) {
  const int max_e = mix_max_elems(dbl), max_t = mix_max_threads(dbl);
  const size_t elem = dbl ? 16 : 8;
  MixGeom m{};
  if (f.nst > kMixStages) return m;
  m.nst = f.nst;
  // threads a line needs when each may hold E elements: one per E / R
  // butterflies, above 17 one per chunk of E / 2 output pairs
  auto chunks = [&](int R, int E) { return ((R + 1) / 2 + E / 2 - 1) / (E / 2); };
  auto threads_for = [&](int E) {
    int t = 1;
    for (int s = 0; s < f.nst; ++s) {
      const int R = f.st[s].radix, nr = f.n / R, q = R > E ? 1 : E / R;
      t = std::max(t, R > 17 ? nr * chunks(R, E == 16 ? max_e : E) : (nr + q - 1) / q);
    }
    return t;
  };
  if (!inter) want = 1;
  else if (!want) want = int(128 / elem);
  // 16 elements per thread; more where a group would not fit its threads
  // otherwise, fewer while the launch leaves SIMDs without a wave.  Two (a lone
  // output pair of a prime above 17) only for an eighth of that: 400 lines of 529
  // complex128, 110000 threads instead of 55000, 16.5 -> 23.3 us
  m.T = threads_for(16);
  if (m.T * want > max_t) m.T = threads_for(max_e);
  const bool full = nlines * m.T >= kFillThreads;
  for (int E : {10, 6, 4, 2})
    if (nlines * m.T < (E == 2 ? kFillThreads / 8 : kFillThreads)) {
      const int t = threads_for(E);
      if (t * want <= max_t && t <= 512) m.T = std::max(m.T, t);
    }
  int ld = f.n, pbi = 1;
  for (int s = 0; s < f.nst; ++s) {
    MixStage &st = m.st[s];
    const int R = f.st[s].radix, ns = f.st[s].ns;
    st.radix = R;
    st.ns = ns;
    st.nr = f.n / R;
    if (R > 17) {
      // few lines: as many chunks as there are threads for
      const int c = full ? chunks(R, max_e) : m.T / st.nr;
      st.q = ((R + 1) / 2 + c - 1) / c;
      m.ngen = std::max(m.ngen, f.st[s].genoff + R);
    } else {
      st.q = (st.nr + m.T - 1) / m.T;
    }
    st.pbi = pbi;
    st.rs = st.nr / ns * pbi;
    st.pbo = s == f.nst - 1 ? f.n : pbo[s];
    pbi = st.pbo;
    st.twoff = f.st[s].twoff;
    st.genoff = f.st[s].genoff;
    st.invns = 1.0f / float(ns);
    ld = std::max(ld, f.n / (ns * R) * st.pbo);
  }
  const size_t cap = lds_bytes - size_t(m.ngen) * elem;
  if (m.T > max_t || size_t(ld) * elem > cap) return m;
  int L = 1;
  if (inter) {
    while (L * 2 <= want && L * 2 * m.T <= max_t && size_t(L * 2) * (ld + 32) * elem <= cap) L *= 2;
    // fewer when the groups would leave CUs idle
    while (L > 2 && nlines < int64_t(L) * 512) L /= 2;
    // the places of a wave's lines (G / L of each) fall into different banks:
    // the pitch is an odd multiple of G / L (three elements at a pitch of 33
    // held a CU to 9 waves: 64M complex64, n = 3 283 -> 193 us)
    const int G = dbl ? 16 : 32, slot = L < G ? G / L : 1;
    if (L > 1) ld += ((slot - ld) % (2 * slot) + 2 * slot) % (2 * slot);
  } else if (m.T <= 128) {
    if (m.T <= 16) ld |= 1;  // the places of a wave's lines fall into different banks
    // groups of about 256 threads; among the sizes up to 512 threads the
    // first that leaves under a tenth of its last wave's lanes idle.  Groups
    // of 5 to 7 waves fill the four SIMDs unevenly: lines of 1000 (100
    // threads) in threes / fives, 65536 of them c64 263 / 240 us, 32000 c128
    // 297 / 250; of 600 (40 threads) in eights / sixes 16000 c64 41.6 / 36.5
    // (no more lines than leave every CU two groups, nor than fit: 2730 lines of
    // 1536 double in fives, half of the nines that fill their waves best, 41.4 us,
    // in threes 23.8)
    const int64_t most = std::min({int64_t(kMixLines), int64_t(512 / m.T), nlines / 512,
                                   int64_t(cap / (size_t(ld) * elem))});
    double best = 0;
    for (int64_t l = std::max<int64_t>(1, std::min<int64_t>(192 / m.T, most)); l <= most; ++l) {
      const int t = int(l) * m.T, waves = (t + 63) / 64;
      const double use = double(t) / double(64 * waves) * (waves > 4 && waves < 8 ? 0.9 : 1.0);
      if (use > best + 0.02) {
        best = use;
        L = int(l);
      }
      if (best >= 0.92) break;
    }
  }
  m.L = L;
  while ((1 << m.log2L) < L) ++m.log2L;
  m.ld = ld;
  m.invT = 1.0f / float(m.T);
  return m;
}

// ... of a call's lines.  Interleaved lines of few threads: adjacent lines
// until they fill a wave; 128-byte rows alone leave a wave of 16 (complex128:
// 8) lines of up to 17 elements with as many live lanes.  us for 4M complex64
// / 2M complex128 elements along axis 0, 128-byte rows / one wave / four: n = 3
// 46.8 / 26.6 / 28.9 and 64.3 / 17.4 / 19.1, n = 12 21.6 / 16.7 / 17.6 and 29.0
// / 15.2 / 15.8, n = 24 21.8 / 18.4 / 19.1 and 24.8 / 18.4 / 18.6, n = 61 39.0
// / 38.6 / 54.3 and 60.4 / 38.0 / 57.9.
template <typename Desc>
MixGeom line_geometry(const Desc &f, const int *pbo, bool dbl, int64_t nlines, bool inter, int want,
                      size_t lds_bytes) {
  MixGeom m = mix_geometry(f, pbo, dbl, nlines, inter, want, lds_bytes);
  if (!inter || !m.L) return m;
  const int base = want ? want : (dbl ? 8 : 16);
  want = base;
  while (want * 2 * m.T <= 64) want *= 2;
  return want == base ? m : mix_geometry(f, pbo, dbl, nlines, inter, want, lds_bytes);
}

}  // namespace rfh
