"""Ragged batches at the edges of the tile classes (workgroups of 64 / 256 /
512 / 1024 threads, the LDS each may take), of the one-pass limits of the tuned
LDS budgets, with prime stages, and with even real lengths whose pairs are
transformed as they lie (no pre or post step).  Every job against the oracle;
bar: rel-L2 <= 1e-6 (complex64/float32), <= 1e-13 (complex128/float64)."""
import numpy as np
import pytest
import torch

import rocket_fft_amd as R
from helpers import rel_l2, tol_of
from test_gpu_ragged import expected, make_jobs

pytestmark = pytest.mark.gpu

SETS = {
    "small": [1, 2, 16, 17, 19, 251, 502, 1023, 1024, 1025, 1040],
    "edges": [4080, 4096, 4097, 5120, 5121, 8192, 8193, 9856, 10240, 16384, 20480],
    # even real lengths with a Bluestein half: c2r first, then c2c, r2c
    "halves": [2 * 4099, 2 * 4099, 2 * 4099, 2 * 10007, 2 * 10007, 2 * 10007, 40000, 40000, 40000],
    "odd": [4099, 4099, 4099, 3 * 5003, 3 * 5003, 3 * 5003, 59 * 61, 173 * 59, 173 * 59],
}


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("name", sorted(SETS))
@pytest.mark.parametrize("autotune", [False, True])
def test_ragged_tiles(dtype, name, autotune):
    jobs, host = make_jobs(dtype, SETS[name], np.random.RandomState(len(name)))
    print(f"case ragged tiles {name} {dtype.__name__} autotune={autotune}", flush=True)
    b = R.RaggedBatch(jobs, double=(dtype == np.complex128), autotune=autotune)
    for _ in range(2):  # the second execution finds the temporaries used
        b.execute()
    torch.cuda.synchronize()
    for (kind, fwd, n, _, out, _), w in zip(jobs, expected(host)):
        e = rel_l2(out.cpu().numpy(), w)
        assert e <= tol_of(dtype), f"{kind} n={n} fwd={fwd}: {e:.3e}"
    b.close()


@pytest.mark.parametrize("n", [2 * 4099, 2 * 10007, 1000, 999])
def test_ragged_real_in_place(n):
    """r2c and c2r with input and output in one buffer."""
    rs = np.random.RandomState(n)
    x = rs.standard_normal(n).astype(np.float32)
    buf = torch.zeros(n // 2 + 1, dtype=torch.complex64, device="cuda")
    real = torch.view_as_real(buf).view(-1)[:n]
    real.copy_(torch.from_numpy(x))
    print(f"case ragged real in place n={n}", flush=True)
    b = R.RaggedBatch([("r2c", True, n, real, buf, 1.0)])
    b.execute()
    torch.cuda.synchronize()
    assert rel_l2(buf.cpu().numpy(), np.fft.rfft(x.astype(np.float64))) <= 1e-6
    b.close()
    b = R.RaggedBatch([("c2r", False, n, buf, real, 1.0 / n)])
    b.execute()
    torch.cuda.synchronize()
    assert rel_l2(real.cpu().numpy(), x) <= 2e-6
    b.close()
