"""Host test of the general line kernel's radices and LDS layout
(rocket-fft_amd/csrc/mixgeom.hpp), compiled with g++: for every length that
fits one workgroup, contiguous and interleaved, the radices multiply to the
length, threads and lines stay within the workgroup's limits, every thread's
butterflies stay within its registers, each stage's writes fill every element
of a line exactly once inside the line's LDS, and the next stage's reads find
element j + r N / R of the Stockham order."""
import os
import subprocess
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "rocket-fft_amd", "csrc")

DRIVER = textwrap.dedent(r"""
    #include <cstdio>
    #include <vector>
    #include "mixgeom.hpp"
    using namespace rfh;
    struct St { int radix, ns, twoff, genoff; };
    struct Desc { int n, nst; St st[24]; };
    #define CHECK(c) do { if (!(c)) { std::printf("FAIL %s n=%d dbl=%d inter=%d\n", #c, n, dbl, inter); return 1; } } while (0)

    int main() {
      const size_t lds = 160 * 1024;
      for (int dbl = 0; dbl < 2; ++dbl)
        for (int variant = 0; variant < 4; ++variant)
        for (int n = 1; n <= (dbl ? 4928 : 9856); ++n) {
          const std::vector<int> rad = variant & 1 ? even_radices(uint64_t(n)) : mix_radices(uint64_t(n));
          Desc f{};
          f.n = n;
          f.nst = int(rad.size());
          int pbo[24] = {}, ns = 1, big = 0, inter = 0;
          for (int s = 0; s < f.nst; ++s) {
            f.st[s] = St{rad[s], ns, 0, 0};
            pbo[s] = block_pitch(ns * rad[s], ns, dbl);
            ns *= rad[s];
            big = std::max(big, rad[s]);
          }
          CHECK(ns == n);
          if (big > 512) continue;  // such primes run as Bluestein
          for (inter = 0; inter < 2; ++inter) {
            if (inter && n > 1216) continue;
            const int want = inter ? (dbl ? 4 : 8) : 0;
            const MixGeom m = mix_geometry(f, pbo, dbl, variant & 2 ? 3 : 1 << 20, inter, want, lds);
            CHECK(m.L >= 1 && m.L * m.T <= mix_max_threads(dbl) && m.L <= kMixLines);
            CHECK(!inter || (m.L == (variant & 2 ? 2 : want) && m.L == 1 << m.log2L));
            CHECK(size_t(m.L * m.ld + m.ngen) * (dbl ? 16 : 8) <= lds && m.ld >= n);
            std::vector<int> at(m.ld);  // which Stockham element a slot holds
            for (int i = 0; i < n; ++i) at[i] = i;
            for (int s = 0; s < f.nst; ++s) {
              const MixStage &st = m.st[s];
              const int R = st.radix;
              if (R <= 17) CHECK(st.q * R <= mix_max_elems(dbl) && st.q * m.T >= st.nr);
              else CHECK(2 * st.q <= mix_max_elems(dbl) && m.T / st.nr * st.q >= (R + 1) / 2);
              if (s > 0 || R > 17)
                for (int j = 0; j < st.nr; ++j)
                  for (int r = 0; r < R; ++r) {
                    const int slot = j / st.ns * st.pbi + j % st.ns + r * st.rs;
                    CHECK(slot < m.ld && at[slot] == j + r * st.nr);
                  }
              std::vector<int> out(m.ld, -1), seen(n, 0);
              for (int j = 0; j < st.nr; ++j)
                for (int r = 0; r < R; ++r) {
                  const int b = j / st.ns, k = j % st.ns;
                  const int slot = b * st.pbo + k + r * st.ns, el = b * st.ns * R + k + r * st.ns;
                  CHECK(slot < m.ld && out[slot] == -1 && !seen[el]++);
                  out[slot] = el;
                }
              at = out;
            }
            for (int i = 0; i < n && f.nst; ++i) CHECK(at[i] == i);  // natural order at the end
          }
        }
      std::printf("OK\n");
      return 0;
    }
""")


def test_mix_geometry(tmp_path):
    src = tmp_path / "geom.cpp"
    exe = tmp_path / "geom"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", f"-I{CSRC}", str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout + r.stderr
