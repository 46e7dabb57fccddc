"""Line sets of any number of groups run: a launch holds at most 2^31 - 1
threads, larger sets take several.  Host: the slices of mixgeom.hpp for tens
of millions of short interleaved lines and millions of long contiguous ones
cover every group once, in order, in as few launches as hold them.  GPU: a
short axis of 34 million lines, and 2^31 contiguous lines in two launches (51
GB, in place), on both sides of every seam.  Bar: rel-L2 <= 1e-6."""
import subprocess
import textwrap

import numpy as np
import pytest

import rocket_fft_amd as R
from helpers import rel_l2
from test_mix_geometry import CSRC

DRIVER = textwrap.dedent(r"""
    #include <cstdio>
    #include "mixgeom.hpp"
    using namespace rfh;
    struct St { int radix, ns, twoff, genoff; };
    struct Desc { int n, nst; St st[24]; };

    int main(int, char **) {
      struct { int n; bool dbl, inter; int64_t lines; } sets[] = {
          {3, false, true, 40000000},   {3, true, true, 25000000},    {2, true, true, 60000000},
          {24, false, true, 30000000},  {2100, false, false, 3000000}, {9856, false, false, 5000000},
          {4000, true, false, 4000000}, {3, false, false, 3000000000}, {7, true, false, 1}};
      for (auto &c : sets) {
        const std::vector<int> rad = mix_radices(uint64_t(c.n));
        Desc f{};
        f.n = c.n;
        int pbo[24] = {}, ns = 1;
        for (int R : rad) {
          f.st[f.nst] = St{R, ns, 0, 0};
          pbo[f.nst++] = block_pitch(ns * R, ns, c.dbl);
          ns *= R;
        }
        const MixGeom m = mix_geometry(f, pbo, c.dbl, c.lines, c.inter, 0, 160 * 1024);
        const int64_t groups = (c.lines + m.L - 1) / m.L;
        const int threads = (m.L * m.T + 63) / 64 * 64;
        int64_t at = 0, launches = 0;
        for_launches(groups, threads, [&](int64_t first, int64_t count) {
          if (first != at || count < 1 || count * threads > 0x7fffffff) at = -1;
          at += count;
          ++launches;
        });
        const int64_t most = 0x7fffffff / threads;
        if (m.L < 1 || at != groups || launches != (groups + most - 1) / most) {
          std::printf("FAIL n=%d\n", c.n);
          return 1;
        }
      }
      std::printf("OK\n");
      return 0;
    }
""")


def test_launch_slices(tmp_path):
    src, exe = tmp_path / "slices.cpp", tmp_path / "slices"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", f"-I{CSRC}", str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout + r.stderr


@pytest.mark.gpu
def test_short_axis_of_many_lines():
    import torch
    lines = 34_000_000
    print(f"case axis 0 of (3, {lines})", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn((3, lines), dtype=torch.complex64, device="cuda", generator=g)
    y = torch.empty_like(x)
    R.c2c(x, y, np.array([0]), True, 1.0)
    for at in (0, lines // 2, lines - 4096):
        want = np.fft.fft(x[:, at:at + 4096].cpu().numpy().astype(np.complex128), axis=0)
        assert rel_l2(y[:, at:at + 4096].cpu().numpy(), want) <= 1e-6


@pytest.mark.gpu
def test_lines_of_several_launches():
    import torch
    lines = (1 << 31) + 1000
    if torch.cuda.mem_get_info()[0] < 24 * lines + (8 << 30):
        pytest.skip("needs 60 GB of device memory")
    print(f"case {lines} lines of 3", flush=True)
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.empty((lines, 3), dtype=torch.complex64, device="cuda")
    block = torch.randn((1 << 20, 3), dtype=torch.complex64, device="cuda", generator=g)
    for lo in range(0, lines, 1 << 20):
        x[lo:lo + (1 << 20)] = block[:min(1 << 20, lines - lo)]
    # the seam of groups of 64 .. 256 lines in 64 .. 256 threads lies among the
    # last 2000 lines before 2^31
    spots = (0, lines // 2, (1 << 31) - 4096, lines - 4096)
    want = [np.fft.fft(x[at:at + 4096].cpu().numpy().astype(np.complex128), axis=1)
            for at in spots]
    R.c2c(x, x, np.array([1]), True, 1.0)
    for at, w in zip(spots, want):
        assert rel_l2(x[at:at + 4096].cpu().numpy(), w) <= 1e-6
    del x
    torch.cuda.empty_cache()
