"""Lines that fit one workgroup with one LDS buffer but not with two: from 32
contiguous lines on they run in one pass (one line per workgroup), below in two
or three.  Host: the geometry driver of test_mix_geometry over those lengths.
GPU: the shortest and longest lengths of both routes against the oracle, few
lines (passes) and many (one pass), plain, in place, strided and rolled.  Bar:
rel-L2 <= 1e-6 (complex64), <= 1e-13 (complex128)."""
import subprocess

import numpy as np
import pytest

import rocket_fft_amd as R
from helpers import oracle_out, rel_l2, tol_of
from test_mix_geometry import CSRC, DRIVER

WHOLE = [(9900, np.complex64), (16384, np.complex64), (17000, np.complex64), (5003, np.complex64),
         (5000, np.complex128), (8192, np.complex128), (9600, np.complex128),
         (4099, np.complex128)]


def test_whole_line_geometry(tmp_path):
    src, exe = tmp_path / "geom.cpp", tmp_path / "geom"
    drv = DRIVER.replace("for (int n = 1; n <= (dbl ? 4928 : 9856); ++n)",
                         "for (int n = (dbl ? 4929 : 9857); n <= (dbl ? 10240 : 20480); ++n)")
    drv = drv.replace("if (big > 512) continue;", "if (big > 17) continue;")
    drv = drv.replace("CHECK(m.L >= 1 &&", "if (m.L == 0) continue;\n            CHECK(m.L == 1 &&")
    assert drv.count("if (m.L == 0) continue;") == 1 and "big > 17" in drv and "4929" in drv
    src.write_text(drv)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", f"-I{CSRC}", str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout + r.stderr


def _lines(rs, shape, dtype):
    return (rs.standard_normal(shape) + 1j * rs.standard_normal(shape)).astype(dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("n,dtype", WHOLE)
@pytest.mark.parametrize("lines", [31, 33])
def test_whole_lines(n, dtype, lines):
    import torch
    rs = np.random.RandomState(n + lines)
    x = _lines(rs, (lines, n), dtype)
    print(f"case whole lines {lines} x {n} {dtype.__name__}", flush=True)
    for fwd, fct in ((True, 1.0), (False, 1.0 / n)):
        want = oracle_out("c2c", x, x, np.array([1]), fwd, fct)
        t = torch.from_numpy(x).cuda()
        out = torch.zeros_like(t)
        R.c2c(t, out, np.array([1]), fwd, fct)
        assert rel_l2(out.cpu().numpy(), want) <= tol_of(dtype)
        wide = torch.zeros((lines, 2 * n), dtype=t.dtype, device="cuda")
        wide[:, ::2] = t  # every other element
        R.c2c(wide[:, ::2], wide[:, 1::2], np.array([1]), fwd, fct)
        assert torch.equal(wide[:, 1::2], out) and torch.equal(wide[:, ::2], t)
        R.c2c(t, t, np.array([1]), fwd, fct)  # in place
        assert torch.equal(t, out)


@pytest.mark.gpu
@pytest.mark.parametrize("n,dtype", [(16384, np.complex64), (4099, np.complex128)])
def test_whole_lines_rolled(n, dtype):
    """Fused rolls of lines in one pass: bit for bit the roll of the plain transform."""
    import torch
    x = _lines(np.random.RandomState(n), (33, n), dtype)
    t = torch.from_numpy(x).cuda()
    for si, so in ((-(n // 2), n // 2), (7, -1)):
        got, plain = torch.zeros_like(t), torch.zeros_like(t)
        assert R.c2c_shifted(t, got, np.array([1]), True, 1.0, [si], [so])
        R.c2c(torch.roll(t, si, 1), plain, np.array([1]), True, 1.0)
        assert torch.equal(got, torch.roll(plain, so, 1))


@pytest.mark.gpu
@pytest.mark.parametrize("first,then", [(33, 3), (3, 33)])
def test_whole_lines_captured_with_the_other_plan(first, then):
    """A length warmed with few lines is captured with many, and the other way
    round: a capture builds no plan, it takes the one there is."""
    import torch
    n = {33: 12000, 3: 12500}[first]  # lengths of its own: no plan of either kind yet
    g = torch.Generator(device="cuda").manual_seed(n)
    big = torch.randn((64, 1 << 16), dtype=torch.complex64, device="cuda", generator=g)
    x = torch.randn((then, n), dtype=torch.complex64, device="cuda", generator=g)
    y = torch.zeros_like(x)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        R.c2c(big, big, np.array([1]), True, 1.0)  # the stream's workspace
        w = torch.randn((first, n), dtype=torch.complex64, device="cuda")
        R.c2c(w, w, np.array([1]), True, 1.0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        R.c2c(x, y, np.array([1]), True, 1.0)
    want = np.fft.fft(x.cpu().numpy().astype(np.complex128), axis=1)
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert rel_l2(y.cpu().numpy(), want) <= 1e-6
    z = torch.zeros_like(x)
    R.c2c_noalloc(x, z, np.array([1]), True, 1.0)
    torch.cuda.synchronize()
    assert torch.equal(z, y)
