"""Real-to-real lines and the plan cache.  A DCT / DST / Hartley call captured
after only a complex transform of its work length has run takes that length's
plan, its factors computed.  The plans of such lines are kept in a cache
directory and read back.  Against scipy in FP64, rel-L2 <= 1e-6 / 1e-13."""
import numpy as np
import pytest
import scipy.fft

import rocket_fft_amd as R
from helpers import rel_l2, tol_of

pytestmark = pytest.mark.gpu

# (call, work length of a line of n, reference)
CALLS = [("dct2", lambda n: n, lambda x: scipy.fft.dct(x, 2, axis=1)),
         ("dct3", lambda n: n, lambda x: scipy.fft.dct(x, 3, axis=1)),
         ("dst4", lambda n: 2 * n, lambda x: scipy.fft.dst(x, 4, axis=1)),
         ("dct1", lambda n: 2 * (n - 1), lambda x: scipy.fft.dct(x, 1, axis=1)),
         ("hartley", lambda n: n,
          lambda x: np.fft.fft(x, axis=1).real + np.fft.fft(x, axis=1).imag)]


def call(kind, x, y):
    if kind == "hartley":
        return R.r2r_separable_hartley(x, y, np.array([1]), 1.0)
    f = R.dct if kind[:3] == "dct" else R.dst
    return f(x, y, np.array([1]), int(kind[3]), 1.0, False)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 54, 243, 512])
@pytest.mark.parametrize("kind,work,ref", CALLS)
def test_captured_after_the_complex_plan(kind, work, ref, n, dtype):
    import torch
    if kind == "dct1" and n == 1:
        pytest.skip("needs two points")
    print(f"case capture {kind} {n} {dtype.__name__}", flush=True)
    R.plan_cache(None, clear_memory=True)  # no plan of either kind
    a = np.random.RandomState(n).standard_normal((5, n)).astype(dtype)
    x = torch.from_numpy(a).cuda()
    y = torch.zeros_like(x)
    m = work(n)
    w = torch.randn((2, m), dtype=torch.complex64 if dtype == np.float32 else torch.complex128,
                    device="cuda")
    s = torch.cuda.Stream()
    big = torch.zeros((64, 1 << 16), dtype=torch.complex128, device="cuda")
    with torch.cuda.stream(s):
        R.c2c(big, big, np.array([1]), True, 1.0)  # the stream's workspace
        R.c2c(w, w, np.array([1]), True, 1.0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        call(kind, x, y)
    want = ref(a.astype(np.float64))
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert rel_l2(y.cpu().numpy(), want) <= tol_of(dtype)
    call(kind, x, y)  # now with its own plan
    assert rel_l2(y.cpu().numpy(), want) <= tol_of(dtype)


def test_real_to_real_plans_in_the_cache_directory(tmp_path):
    import torch
    R.plan_cache(str(tmp_path), clear_memory=True)
    try:
        x = torch.rand((3, 361), dtype=torch.float64, device="cuda")
        first = []
        print("case real-to-real plans on disk", flush=True)
        for kind, _, _ in CALLS:
            y = torch.empty_like(x)
            call(kind, x, y)
            first.append(y)
        files = sorted(p.name for p in tmp_path.iterdir())
        # the two types with factors of a work line of 361 share a plan
        assert len(files) == 4 and all("_r2r_" in f for f in files), files
        R.plan_cache(str(tmp_path), clear_memory=True)
        h0, w0 = R.plan_cache_stats()
        for (kind, _, _), want in zip(CALLS, first):
            y = torch.empty_like(x)
            call(kind, x, y)
            assert torch.equal(y, want)
        assert R.plan_cache_stats() == (h0 + 4, w0)
    finally:
        R.plan_cache(None, clear_memory=True)
