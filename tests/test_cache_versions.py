"""What earlier builds left in the cache directories is not used: plan records
without this build's schedule version, and tuning results of other kernels, are
ignored, built or timed again, and rewritten or appended."""
import struct

import numpy as np
import pytest

import rocket_fft_amd as R
from test_plan_cache import fnv1a64

VERSION = 2


def without_version(f):
    """The record of a build that wrote no schedule version."""
    body = f[:-12]
    return body + struct.pack("<Q", fnv1a64(body))


def test_plan_record_names_its_schedule(tmp_path):
    for real in (False, True):
        path = tmp_path / f"plan{real}.bin"
        assert R.plan_record_roundtrip(1000, False, 131072, False, real, path=str(path)) == 0
        f = path.read_bytes()
        assert struct.unpack("<I", f[-12:-8])[0] == VERSION


@pytest.mark.gpu
def test_plan_record_of_an_earlier_build_is_rebuilt(tmp_path):
    import torch
    R.plan_cache(str(tmp_path), clear_memory=True)
    try:
        x = torch.randn((3, 1000), dtype=torch.complex64, device="cuda")
        a, b = torch.empty_like(x), torch.empty_like(x)
        print("case plan record without a schedule version", flush=True)
        R.c2c(x, a, np.array([1]), True, 1.0)
        (path,) = tmp_path.iterdir()
        good = path.read_bytes()
        path.write_bytes(without_version(good))
        R.plan_cache(str(tmp_path), clear_memory=True)
        h0, w0 = R.plan_cache_stats()
        R.c2c(x, b, np.array([1]), True, 1.0)
        assert R.plan_cache_stats() == (h0, w0 + 1)
        assert path.read_bytes() == good and torch.equal(a, b)
    finally:
        R.plan_cache(None)


def old_key(sig):
    """Key of a tuning line before it held a version."""
    m = (1 << 64) - 1
    h1, h2 = 1469598103934665603, 0x9E3779B97F4A7C15
    for v in sig:
        for b in range(8):
            h1 = ((h1 ^ ((v >> (8 * b)) & 0xFF)) * 1099511628211) & m
        h2 ^= (v + 0x9E3779B97F4A7C15 + (h2 << 6) + (h2 >> 2)) & m
        h2 = (h2 * 0xFF51AFD7ED558CCD) & m
    return h1, h2, len(sig)


@pytest.mark.gpu
def test_tuning_line_of_an_earlier_build_is_not_used(tmp_path):
    import torch
    ns = [64, 1000, 4099, 300]
    jobs = [("c2c", True, n, torch.randn(n, dtype=torch.complex64, device="cuda"),
             torch.empty(n, dtype=torch.complex64, device="cuda"), 1.0) for n in ns]
    R.set_tune_cache(tmp_path, clear_memory=True)
    try:
        print("case tuning line without a version", flush=True)
        R.RaggedBatch(jobs, autotune=True)
        (path,) = tmp_path.iterdir()
        h1, h2, n = old_key([0] + ns)  # complex64, then (kind << 60) ^ length of every job
        path.write_text(f"rfh1 {h1:016x} {h2:016x} {n} 65536 512\n")
        R.set_tune_cache(tmp_path, clear_memory=True)
        assert R.RaggedBatch(jobs, autotune=True).info()["autotuned"] == 1
        assert len(path.read_text().splitlines()) == 2
        R.set_tune_cache(tmp_path, clear_memory=True)
        assert R.RaggedBatch(jobs, autotune=True).info()["autotuned"] == 3
    finally:
        R.set_tune_cache(None)
