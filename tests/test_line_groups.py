"""Groups of short lines.  Host: an interleaved group of short lines fills more
than half of its waves' lanes and stays inside the workgroup and its LDS, at
every length to 100; a contiguous group fills its waves as well as any smaller
one.  GPU: short lengths along axis 0 with enough lines for
whole waves, the last group a part of one, against numpy in FP64, forward and
inverse, complex, real and back.  Bar: rel-L2 <= 1e-6 / 1e-13."""
import subprocess
import textwrap

import numpy as np
import pytest

import rocket_fft_amd as R
from helpers import RTYPE, rel_l2, tol_of
from test_mix_geometry import CSRC

DRIVER = textwrap.dedent(r"""
    #include <cstdio>
    #include "mixgeom.hpp"
    using namespace rfh;
    struct St { int radix, ns, twoff, genoff; };
    struct Desc { int n, nst; St st[24]; };

    int main() {
      for (int dbl = 0; dbl < 2; ++dbl)
        for (int n = 1; n <= 100; ++n)
          for (int want : {0, 4, 16})
            for (int64_t lines : {int64_t(5), int64_t(3000), int64_t(1) << 20}) {
              const std::vector<int> rad = mix_radices(uint64_t(n));
              Desc f{};
              f.n = n;
              int pbo[24] = {}, ns = 1, gen = 0;
              for (int R : rad) {
                f.st[f.nst] = St{R, ns, 0, gen};
                if (R > 17) gen += R;
                pbo[f.nst++] = block_pitch(ns * R, ns, dbl);
                ns *= R;
              }
              const MixGeom m = line_geometry(f, pbo, dbl, lines, true, want, 160 * 1024);
              const int t = m.L * m.T, lanes = (t + 63) / 64 * 64;
              bool ok = m.L >= 2 && m.L == 1 << m.log2L && m.L <= kMixLines && t <= mix_max_threads(dbl);
              ok = ok && size_t(m.L * m.ld + m.ngen) * (dbl ? 16 : 8) <= 160 * 1024;
              if (lines == 1 << 20) ok = ok && 2 * t > lanes;
              // one stage: a line takes its elements and a pitch that spreads the banks
              const int G = dbl ? 16 : 32, slot = m.L < G ? G / m.L : 1;
              if (m.nst < 2) ok = ok && m.ld < n + 2 * slot && m.ld % (2 * slot) == slot % (2 * slot);
              if (!ok) {
                std::printf("FAIL n=%d dbl=%d want=%d: %d lines of %d threads\n", n, dbl, want, m.L, m.T);
                return 1;
              }
            }
      // contiguous lines: a set too small for the group that fills its waves best
      // takes the best of those it has two a CU of, not a part of that group
      for (int dbl = 0; dbl < 2; ++dbl)
        for (int n = 2; n <= 1000; ++n)
          for (int64_t lines : {int64_t(600), int64_t(2730), int64_t(9000)}) {
            const std::vector<int> rad = even_radices(uint64_t(n));
            Desc f{};
            f.n = n;
            int pbo[24] = {}, ns = 1;
            for (int R : rad) {
              f.st[f.nst] = St{R, ns, 0, 0};
              pbo[f.nst++] = block_pitch(ns * R, ns, dbl);
              ns *= R;
            }
            if (rad.back() > 17) continue;
            const MixGeom m = line_geometry(f, pbo, dbl, lines, false, 0, 160 * 1024);
            auto use = [&](int l) {
              const int t = l * m.T, waves = (t + 63) / 64;
              return double(t) / (64 * waves) * (waves > 4 && waves < 8 ? 0.9 : 1.0);
            };
            bool ok = m.L >= 1 && (m.L == 1 || m.L * 512 <= lines) && m.L * m.T <= 1024;
            for (int l = std::max(1, 192 / m.T); l < m.L; ++l) ok = ok && use(l) <= use(m.L);
            if (!ok) {
              std::printf("FAIL n=%d dbl=%d lines=%d: %d lines of %d\n", n, dbl, int(lines), m.L, m.T);
              return 1;
            }
          }
      std::printf("OK\n");
      return 0;
    }
""")


def test_short_groups_fill_their_waves(tmp_path):
    src, exe = tmp_path / "groups.cpp", tmp_path / "groups"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", f"-I{CSRC}", str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout + r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n", [2, 3, 5, 6, 9, 12, 17, 19, 24, 31, 34, 61])
def test_short_axis_groups(n, dtype):
    import torch
    lines = 64 * 512 + 37
    print(f"case axis 0 of ({n}, {lines}) {dtype.__name__}", flush=True)
    rs = np.random.RandomState(n)
    z = (rs.standard_normal((n, lines)) + 1j * rs.standard_normal((n, lines))).astype(dtype)
    r = rs.standard_normal((n, lines)).astype(RTYPE[dtype])
    t, y = torch.from_numpy(z).cuda(), torch.empty((n, lines), dtype=getattr(torch, dtype.__name__), device="cuda")
    ax = np.array([0])
    for fwd, f in ((True, np.fft.fft), (False, np.fft.ifft)):
        R.c2c(t, y, ax, fwd, 1.0 if fwd else 1.0 / n)
        assert rel_l2(y.cpu().numpy(), f(z.astype(np.complex128), axis=0)) <= tol_of(dtype)
    half = torch.empty((n // 2 + 1, lines), dtype=y.dtype, device="cuda")
    back = torch.from_numpy(np.zeros_like(r)).cuda()
    R.r2c(torch.from_numpy(r).cuda(), half, ax, True, 1.0)
    assert rel_l2(half.cpu().numpy(), np.fft.rfft(r.astype(np.float64), axis=0)) <= tol_of(dtype)
    R.c2r(half, back, ax, False, 1.0 / n)
    assert rel_l2(back.cpu().numpy(), r) <= 2 * tol_of(dtype)
    R.c2c(t, t, ax, False, 1.0 / n)  # in place
    assert torch.equal(t, y)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("lines", [3, 257 * 9 + 1, 512 * 64 + 5])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 7, 9, 10, 12, 17, 18, 19, 24, 30, 37, 48, 62, 96])
def test_short_rows(n, lines, dtype):
    """Contiguous rows, groups of one line and of many, the last group a part
    of one; a padded output keeps its gaps."""
    import scipy.fft
    import torch
    ax = np.array([1])
    print(f"case rows ({lines}, {n}) {dtype.__name__}", flush=True)
    rs = np.random.RandomState(100 + n)
    z = (rs.standard_normal((lines, n)) + 1j * rs.standard_normal((lines, n))).astype(dtype)
    r = rs.standard_normal((lines, n)).astype(RTYPE[dtype])
    t, x = torch.from_numpy(z).cuda(), torch.from_numpy(r).cuda()
    tol = tol_of(dtype)
    for fwd, f in ((True, np.fft.fft), (False, np.fft.ifft)):
        wide = torch.full((lines, n + 1), 7, dtype=t.dtype, device="cuda")
        R.c2c(t, wide[:, :n], ax, fwd, 1.0 if fwd else 1.0 / n)
        assert rel_l2(wide[:, :n].cpu().numpy(), f(z.astype(np.complex128), axis=1)) <= tol
        assert bool((wide[:, n] == 7).all())
    u = t.clone()
    R.c2c(u, u, ax, False, 1.0 / n)  # in place
    assert torch.equal(u, wide[:, :n])
    half = torch.full((lines, n // 2 + 2), 7, dtype=t.dtype, device="cuda")
    R.r2c(x, half[:, :-1], ax, True, 1.0)
    assert rel_l2(half[:, :-1].cpu().numpy(), np.fft.rfft(r.astype(np.float64), axis=1)) <= tol
    assert bool((half[:, -1] == 7).all())
    back = torch.full((lines, n + 1), 7, dtype=x.dtype, device="cuda")
    R.c2r(half[:, :-1], back[:, :n], ax, False, 1.0 / n)
    assert rel_l2(back[:, :n].cpu().numpy(), r) <= 2 * tol and bool((back[:, n] == 7).all())
    y = torch.empty_like(x)
    for kind in (1, 2, 3, 4):
        if kind == 1 and n < 2:
            continue
        R.dct(x, y, ax, kind, 1.0, False)
        assert rel_l2(y.cpu().numpy(), scipy.fft.dct(r.astype(np.float64), kind, axis=1)) <= tol
    R.r2r_separable_hartley(x, y, ax, 1.0)
    f = np.fft.fft(r.astype(np.float64), axis=1)
    assert rel_l2(y.cpu().numpy(), f.real + f.imag) <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n", [19, 23, 38, 61, 97, 122, 194, 361, 437, 529, 1147, 1220, 1681])
def test_prime_radices_few_and_many_lines(n, dtype):
    """Lines with a prime above 17: one output pair a thread (few lines), several
    (more of them) and many, rows and columns."""
    import torch
    for lines in (1, 24, 400, 5000):
        print(f"case primes {lines} x {n} {dtype.__name__}", flush=True)
        rs = np.random.RandomState(n + lines)
        z = (rs.standard_normal((lines, n)) + 1j * rs.standard_normal((lines, n))).astype(dtype)
        want = np.fft.fft(z.astype(np.complex128), axis=1)
        t = torch.from_numpy(z).cuda()
        y = torch.empty_like(t)
        R.c2c(t, y, np.array([1]), True, 1.0)
        assert rel_l2(y.cpu().numpy(), want) <= tol_of(dtype)
        c = t.T.contiguous()
        R.c2c(c, c, np.array([0]), True, 1.0)
        assert rel_l2(c.T.cpu().numpy(), want) <= tol_of(dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n", [3, 6, 9, 12, 17, 24, 30, 37])
def test_short_rows_of_spread_elements(n, dtype):
    """Rows of every third input element to every second output one; what lies
    between the outputs stays."""
    import torch
    lines, ax = 512 * 64 + 5, np.array([1])
    print(f"case spread rows ({lines}, {n}) {dtype.__name__}", flush=True)
    rs = np.random.RandomState(200 + n)
    z = (rs.standard_normal((lines, 3 * n)) + 1j * rs.standard_normal((lines, 3 * n))).astype(dtype)
    r = rs.standard_normal((lines, 3 * n)).astype(RTYPE[dtype])
    t, x = torch.from_numpy(z).cuda()[:, ::3], torch.from_numpy(r).cuda()[:, ::3]
    tol, h = tol_of(dtype), n // 2 + 1
    wide = torch.full((lines, 2 * n), 7, dtype=t.dtype, device="cuda")
    R.c2c(t, wide[:, ::2], ax, False, 1.0 / n)
    assert rel_l2(wide[:, ::2].cpu().numpy(), np.fft.ifft(z[:, ::3].astype(np.complex128), axis=1)) <= tol
    assert bool((wide[:, 1::2] == 7).all())
    half = torch.full((lines, 2 * h), 7, dtype=t.dtype, device="cuda")
    R.r2c(x, half[:, ::2], ax, True, 1.0)
    assert rel_l2(half[:, ::2].cpu().numpy(), np.fft.rfft(r[:, ::3].astype(np.float64), axis=1)) <= tol
    assert bool((half[:, 1::2] == 7).all())
    back = torch.full((lines, 2 * n), 7, dtype=x.dtype, device="cuda")
    R.c2r(half[:, ::2], back[:, ::2], ax, False, 1.0 / n)
    assert rel_l2(back[:, ::2].cpu().numpy(), r[:, ::3]) <= 2 * tol and bool((back[:, 1::2] == 7).all())
    y = torch.empty((lines, n), dtype=x.dtype, device="cuda")
    R.r2r_separable_hartley(x, y, ax, 1.0)
    f = np.fft.fft(r[:, ::3].astype(np.float64), axis=1)
    assert rel_l2(y.cpu().numpy(), f.real + f.imag) <= tol
