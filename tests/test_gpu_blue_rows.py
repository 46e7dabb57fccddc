"""Bluestein lines in three passes with power-of-two rows: forward stages, kernel
product in registers, the inverse transform's stages backwards.  Rows of 8 to
1024 (one, two and three stages), contiguous and interleaved lines, both
directions, more lines than one workgroup takes; against numpy's FP64 FFT, bar
rel-L2 <= 1e-6 (complex64), <= 1e-13 (complex128)."""
import numpy as np
import pytest

import rocket_fft_amd as R
from helpers import rel_l2, tol_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,axis,rows,dtype", [
    (4093, 1, 32, np.complex128), (8191, 1, 64, np.complex64), (16381, 1, 128, np.complex64),
    (131071, 1, 1024, np.complex64), (131071, 1, 1024, np.complex128),
    (1021, 0, 8, np.complex128), (2039, 0, 16, np.complex128), (2039, 0, 16, np.complex64),
    (4093, 0, 32, np.complex64), (10037, 1, 80, np.complex64)])
def test_bluestein_rows(n, axis, rows, dtype):
    import torch
    if axis == 1:
        kind, _, n1, n2 = R.gpu_schedule(n, dtype == np.complex128)
        assert (kind, n1, n2) == (3, 256, rows)
    rs = np.random.RandomState(n)
    shape = (5, n) if axis else (n, 37)
    x = (rs.standard_normal(shape) + 1j * rs.standard_normal(shape)).astype(dtype)
    print(f"case bluestein rows n={n} axis={axis} {dtype.__name__}", flush=True)
    t = torch.from_numpy(x).cuda()
    y = torch.empty_like(t)
    R.c2c(t, y, np.array([axis]), True, 1.0)
    assert rel_l2(y.cpu().numpy(), np.fft.fft(x.astype(np.complex128), axis=axis)) <= tol_of(dtype)
    R.c2c(t, t, np.array([axis]), False, 1.0 / n)  # in place
    assert rel_l2(t.cpu().numpy(), np.fft.ifft(x.astype(np.complex128), axis=axis)) <= tol_of(dtype)
