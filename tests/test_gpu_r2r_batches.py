"""Real-to-real lines at the edges of a thread's batch of loads and stores and of
the threads of a group: one line, a few and many, lengths around 8 elements a
thread, DCT and DST of all four types, contiguous and strided lines.  Against
SciPy's FP64 transform; bar rel-L2 <= 1e-6 (float32), <= 1e-13 (float64)."""
import numpy as np
import pytest
import scipy.fft

import rocket_fft_amd as R
from helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(np.float32, 1e-6), (np.float64, 1e-13)])
@pytest.mark.parametrize("n", [2, 9, 64, 65, 511, 513])
@pytest.mark.parametrize("lines", [1, 5, 700])
def test_r2r_batches(n, lines, dtype, tol):
    import torch
    x = np.random.RandomState(n + lines).standard_normal((lines, n)).astype(dtype)
    t = torch.from_numpy(x).cuda()
    ts = torch.from_numpy(np.ascontiguousarray(x.T)).cuda()
    print(f"case r2r batches {lines} x {n} {dtype.__name__}", flush=True)
    for typ in (1, 2, 3, 4):
        for f, g in ((R.dct, scipy.fft.dct), (R.dst, scipy.fft.dst)):
            want = g(x.astype(np.float64), typ, axis=1)
            y, ys = torch.empty_like(t), torch.empty_like(ts)
            f(t, y, np.array([1]), typ, 1.0, False)
            f(ts, ys, np.array([0]), typ, 1.0, False)
            assert rel_l2(y.cpu().numpy(), want) <= tol, (f.__name__, typ)
            assert rel_l2(ys.cpu().numpy().T, want) <= tol, (f.__name__, typ, "strided")
