"""Performance cases: transforms as programs call them, with their inputs,
the work they cannot do without and their exact results.

Every case names its `kind` of call and the sizes, precision and options of
that call:

  small    one front-end call on a few short lines (latency of one call)
  lines    batched power-of-two lines through the low-level c2c, output
           array kept by the caller
  mixed    batched lines of other lengths, front-end fft / ifft
  prime    batched lines of prime length (Bluestein), low-level c2c
  image    fft2 / ifft2 of a stack of images of any size
  real3d   rfftn of a field and irfftn of its spectrum
  cosine   dctn / dstn and their inverses of an image
  ragged   a RaggedBatch of transforms of uneven lengths, executed once
  host     front-end call on NumPy arrays in host memory

Lines, mixed, prime, real3d, cosine and ragged hold the sizes that bench.py
measures; the others are generic sizes of the same kinds.
"""
import bisect
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "rocket-fft_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

MAX_BYTES = 1 << 30  # of one pass, input and output together (the largest listed case)


def listed():
    return [
        # a single short call in a latency-bound program: one block of samples
        {"name": "small_16x256_c64", "kind": "small", "batch": 16, "n": 256, "double": False,
         "forward": True},
        # long signals, a batch of 2^20-point spectra (the precision configuration)
        {"name": "lines_64x2p20_c64", "kind": "lines", "batch": 64, "n": 1 << 20,
         "double": False, "forward": True},
        # many medium lines (the precision configuration's second array)
        {"name": "lines_16384x4096_c64", "kind": "lines", "batch": 16384, "n": 4096,
         "double": False, "forward": True},
        # double precision and the inverse direction on a medium batch
        {"name": "lines_1024x4096_c128", "kind": "lines", "batch": 1024, "n": 4096,
         "double": True, "forward": False},
        # decimal block length, a large batch
        {"name": "mixed_4096x1000_c64", "kind": "mixed", "batch": 4096, "n": 1000,
         "double": False, "forward": True},
        # NumPy arrays in host memory, as a program without GPU code of its own calls it
        {"name": "host_256x1000_c128", "kind": "host", "batch": 256, "n": 1000,
         "double": True, "forward": True},
        # prime lengths: one that pads into one workgroup's memory, one far beyond it
        {"name": "prime_256x4099_c128", "kind": "prime", "batch": 256, "n": 4099,
         "double": True, "forward": True},
        {"name": "prime_256x65537_c64", "kind": "prime", "batch": 256, "n": 65537,
         "double": False, "forward": True},
        # spectra of a stack of video-sized frames: both axes, one of them strided
        {"name": "image_8x1080x1920_c64", "kind": "image", "batch": 8, "h": 1080, "w": 1920,
         "double": False, "forward": True},
        # a field solver's round trip: real field to half spectrum and back
        {"name": "real3d_256_f32", "kind": "real3d", "a": 256, "b": 256, "c": 256,
         "double": False},
        # DCT-II of one image, orthonormal
        {"name": "dct2_512x512_f64", "kind": "cosine", "h": 512, "w": 512, "type": 2,
         "cosine": True, "inverse": False, "ortho": True, "double": True},
        # a queue of unrelated transforms of uneven lengths
        {"name": "ragged_4096", "kind": "ragged", "jobs": 4096, "lengths": 5},
    ]


# ------------------------------------------------------------------ drawing

def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _is_prime(n):
    return n > 1 and all(n % d for d in range(2, int(math.isqrt(n)) + 1))


def _batch(rng, n, double, lo_elems, hi_elems):
    """Lines of n elements holding lo_elems .. hi_elems elements in all."""
    top = min(hi_elems, MAX_BYTES // (32 if double else 16))
    elems = _log(rng, max(n, min(lo_elems, top)), max(n, top))
    return max(1, elems // n)


def draw(rng):
    kind = rng.choice(("small", "lines", "lines", "mixed", "mixed", "prime", "image", "image",
                       "real3d", "cosine", "ragged", "host"))
    double = rng.random() < 0.4
    forward = rng.random() < 0.6
    if kind == "small":
        return {"kind": kind, "batch": _log(rng, 1, 64), "n": _log(rng, 16, 4096),
                "double": double, "forward": forward}
    if kind == "lines":
        n = 1 << rng.randint(6, 20)
        return {"kind": kind, "batch": _batch(rng, n, double, 1 << 18, 1 << 26), "n": n,
                "double": double, "forward": forward}
    if kind == "mixed":
        n = _log(rng, 60, 12000)
        if rng.random() < 0.6:  # a good length, as programs pad to
            n = _good(n, False)
        return {"kind": kind, "batch": _batch(rng, n, double, 1 << 17, 1 << 23), "n": n,
                "double": double, "forward": forward}
    if kind == "prime":
        n = _log(rng, 211, 70000)
        while not _is_prime(n):
            n += 1
        return {"kind": kind, "batch": _batch(rng, n, double, 1 << 17, 1 << 23), "n": n,
                "double": double, "forward": forward}
    if kind == "image":
        return {"kind": kind, "batch": rng.randint(1, 8), "h": _log(rng, 128, 2048),
                "w": _log(rng, 128, 2048), "double": double, "forward": forward}
    if kind == "real3d":
        a, b, c = (_log(rng, 24, 256) for _ in range(3))
        return {"kind": kind, "a": a, "b": b, "c": c, "double": double}
    if kind == "cosine":
        return {"kind": kind, "h": _log(rng, 48, 1024), "w": _log(rng, 48, 1024),
                "type": rng.randint(1, 4), "cosine": rng.random() < 0.7,
                "inverse": rng.random() < 0.4, "ortho": rng.random() < 0.5, "double": double}
    if kind == "ragged":
        return {"kind": kind, "jobs": _log(rng, 32, 2048), "lengths": rng.randint(1, 1 << 20)}
    return {"kind": "host", "batch": _log(rng, 1, 256), "n": _log(rng, 100, 8000),
            "double": double, "forward": forward}


# ------------------------------------------------------------------- inputs

_SMOOTH = {}


def _good(n, real):
    """Smallest length >= n whose prime factors are at most 11 (5 for real)."""
    if real not in _SMOOTH:
        got = [1]
        for p in (2, 3, 5) if real else (2, 3, 5, 7, 11):
            more = list(got)
            while more:
                more = [v * p for v in more if v * p <= 1 << 18]
                got += more
        _SMOOTH[real] = sorted(got)
    s = _SMOOTH[real]
    return s[bisect.bisect_left(s, n)]


def _ragged_spec(jobs, lengths):
    """(kind, n) of each job: lengths log-uniform in 64 .. 65536, 70% of them
    rounded up to a good length, 60% complex, 40% real."""
    rs = np.random.RandomState(lengths)
    raw = np.exp(rs.uniform(np.log(64), np.log(65536), jobs)).astype(np.int64)
    good = rs.uniform(size=jobs) < 0.7
    c2c = rs.uniform(size=jobs) < 0.6
    spec = []
    for n, g, c in zip(raw, good, c2c):
        n = _good(int(n), not c) if g else int(n)
        spec.append(("c2c" if c else "r2c", n))
    return spec


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _dt(case, real=False):
    if real:
        return torch.float64 if case["double"] else torch.float32
    return torch.complex128 if case["double"] else torch.complex64


def _aligned(count):
    return -(-count // 64) * 64  # every job's line starts on a boundary of its own


def _input(case, seed):
    k = case["kind"]
    if k in ("small", "lines", "mixed", "prime"):
        return torch.randn((case["batch"], case["n"]), dtype=_dt(case), device="cuda",
                           generator=_gen(seed))
    if k == "image":
        return torch.randn((case["batch"], case["h"], case["w"]), dtype=_dt(case),
                           device="cuda", generator=_gen(seed))
    if k == "real3d":
        return torch.randn((case["a"], case["b"], case["c"]), dtype=_dt(case, True),
                           device="cuda", generator=_gen(seed))
    if k == "cosine":
        return torch.rand((case["h"], case["w"]), dtype=_dt(case, True), device="cuda",
                          generator=_gen(seed)) * 2 - 1
    if k == "ragged":  # one float buffer; job i's line starts at offset[i]
        total = sum(_aligned((2 if kind == "c2c" else 1) * n)
                    for kind, n in _ragged_spec(case["jobs"], case["lengths"]))
        return torch.randn(total, dtype=torch.float32, device="cuda", generator=_gen(seed))
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((case["batch"], case["n"], 2),
                            dtype=np.float64 if case["double"] else np.float32)
    return x.view(np.complex128 if case["double"] else np.complex64)[..., 0]


def _ragged_views(case, x, y):
    """(kind, n, input line, output line) of every job in the flat buffers."""
    jobs, xo, yo = [], 0, 0
    for kind, n in _ragged_spec(case["jobs"], case["lengths"]):
        nout = n if kind == "c2c" else n // 2 + 1
        if kind == "c2c":
            line = torch.view_as_complex(x[xo:xo + 2 * n].view(-1, 2))
            xo += _aligned(2 * n)
        else:
            line = x[xo:xo + n]
            xo += _aligned(n)
        jobs.append((kind, n, line, None if y is None else y[yo:yo + nout]))
        yo += _aligned(nout)
    return jobs, yo


# ------------------------------------------------------------- prepare, run

def prepare(case, seed):
    import rocket_fft_amd as R
    import rocket_fft_amd.fft as F
    x = _input(case, seed)
    s = {"case": case, "R": R, "F": F, "x": x}
    if case["kind"] in ("lines", "prime"):
        s["y"] = torch.empty_like(x)
        s["axes"] = np.array([1])
    elif case["kind"] == "ragged":
        s["y"] = torch.zeros(_ragged_views(case, x, None)[1], dtype=torch.complex64,
                             device="cuda")
        jobs, _ = _ragged_views(case, x, s["y"])
        s["batch"] = R.RaggedBatch([(kind, True, n, a, b, 1.0) for kind, n, a, b in jobs])
    return s


def run(state):
    case, F, x = state["case"], state["F"], state["x"]
    k = case["kind"]
    if k in ("small", "mixed", "host"):
        return F.fft(x) if case["forward"] else F.ifft(x)
    if k in ("lines", "prime"):
        fct = 1.0 if case["forward"] else 1.0 / case["n"]
        return state["R"].c2c(x, state["y"], state["axes"], case["forward"], fct)
    if k == "image":
        return F.fft2(x) if case["forward"] else F.ifft2(x)
    if k == "real3d":
        spec = F.rfftn(x)
        s = None if x.shape[-1] % 2 == 0 else tuple(x.shape)  # an odd size has to be named
        return {"spectrum": spec, "field": F.irfftn(spec, s=s)}
    if k == "cosine":
        name = ("i" if case["inverse"] else "") + ("dctn" if case["cosine"] else "dstn")
        return getattr(F, name)(x, type=case["type"], norm="ortho" if case["ortho"] else None)
    state["batch"].execute()
    return state["y"]


# --------------------------------------------------------------------- work

def work(case):
    """Each input read once and each output written once; 5 n log2 n
    operations for a complex line of n, half of that for a real one."""
    k = case["kind"]
    if k == "ragged":
        nbytes = flops = 0.0
        for kind, n in _ragged_spec(case["jobs"], case["lengths"]):
            nbytes += 16 * n if kind == "c2c" else 4 * n + 8 * (n // 2 + 1)
            flops += (5.0 if kind == "c2c" else 2.5) * n * math.log2(n)
        return {"bytes": nbytes, "flops": flops}
    scalar = 8 if case["double"] else 4
    if k == "real3d":
        a, b, c = case["a"], case["b"], case["c"]
        one = scalar * a * b * (c + 2 * (c // 2 + 1))
        return {"bytes": 2 * one, "flops": 2 * 2.5 * a * b * c * math.log2(a * b * c)}
    if k == "cosine":
        n = case["h"] * case["w"]
        return {"bytes": 2 * scalar * n, "flops": 2.5 * n * math.log2(n)}
    if k == "image":
        n, lines = case["h"] * case["w"], case["batch"]
    else:
        n, lines = case["n"], case["batch"]
    return {"bytes": 4 * scalar * lines * n, "flops": 5.0 * lines * n * math.log2(n)}


# -------------------------------------------------------------------- exact

def _trig(n, kind, cosine):
    """The n x n matrix of the unnormalised DCT / DST of a type (rows:
    outputs), float64."""
    j = torch.arange(n, dtype=torch.float64, device="cuda")[None, :]
    k = torch.arange(n, dtype=torch.float64, device="cuda")[:, None]

    def angle(num, den):  # pi num / den, reduced exactly
        return torch.remainder(num, 2 * den) * (math.pi / den)

    if cosine:
        if kind == 1:
            m = 2 * torch.cos(angle(j * k, n - 1))
            m[:, 0] /= 2
            m[:, n - 1] /= 2
        elif kind == 2:
            m = 2 * torch.cos(angle(k * (2 * j + 1), 2 * n))
        elif kind == 3:
            m = 2 * torch.cos(angle(j * (2 * k + 1), 2 * n))
            m[:, 0] /= 2
        else:
            m = 2 * torch.cos(angle((2 * k + 1) * (2 * j + 1), 4 * n))
    elif kind == 1:
        m = 2 * torch.sin(angle((j + 1) * (k + 1), n + 1))
    elif kind == 2:
        m = 2 * torch.sin(angle((k + 1) * (2 * j + 1), 2 * n))
    elif kind == 3:
        m = 2 * torch.sin(angle((j + 1) * (2 * k + 1), 2 * n))
        m[:, n - 1] /= 2
    else:
        m = 2 * torch.sin(angle((2 * k + 1) * (2 * j + 1), 4 * n))
    return m


def _exact_cosine(case, x):
    t = {2: 3, 3: 2}.get(case["type"], case["type"]) if case["inverse"] else case["type"]
    y = x.to(torch.float64)
    scale = 1.0
    for axis in (0, 1):
        n = y.shape[axis]
        m = _trig(n, t, case["cosine"])
        if case["ortho"]:  # orthonormal scaling of the ends, as the front-end defines it
            if t == 1 and case["cosine"]:
                m[:, 0] *= math.sqrt(2)
                m[:, n - 1] *= math.sqrt(2)
                m[0] /= math.sqrt(2)
                m[n - 1] /= math.sqrt(2)
            elif t == 2:
                m[0] /= math.sqrt(2)
            elif t == 3:
                m[:, 0] *= math.sqrt(2)
        y = m @ y if axis == 0 else y @ m.T
        scale *= 2.0 * (n + ((-1 if case["cosine"] else 1) if t == 1 else 0))
    if case["ortho"]:
        return y / math.sqrt(scale)
    return y / scale if case["inverse"] else y


def exact(case, seed):
    x = _input(case, seed)
    k = case["kind"]
    if k == "cosine":
        return _exact_cosine(case, x)
    if k == "real3d":
        # the inverse has the computed spectrum for its input, not this one:
        # its exact value is the field it came from
        return {"spectrum": torch.fft.rfftn(x.to(torch.float64)), "field": x.to(torch.float64)}
    if k == "image":
        f = torch.fft.fft2 if case["forward"] else torch.fft.ifft2
        return f(x.to(torch.complex128))
    if k == "ragged":
        xh = x.cpu()
        jobs, total = _ragged_views(case, xh, None)
        y, yo = np.zeros(total, dtype=np.complex128), 0
        for kind, n, line, _ in jobs:
            a = line.numpy()
            want = (np.fft.fft(a.astype(np.complex128)) if kind == "c2c"
                    else np.fft.rfft(a.astype(np.float64)))
            y[yo:yo + want.size] = want
            yo += _aligned(want.size)
        return y
    if k == "host":
        return (np.fft.fft if case["forward"] else np.fft.ifft)(x.astype(np.complex128))
    out, step = torch.empty(x.shape, dtype=torch.complex128, device="cuda"), \
        max(1, (1 << 24) // case["n"])
    f = torch.fft.fft if case["forward"] else torch.fft.ifft
    for lo in range(0, x.shape[0], step):
        out[lo:lo + step] = f(x[lo:lo + step].to(torch.complex128), dim=1)
    return out
