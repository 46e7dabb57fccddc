"""The host side of a call: every accepted form of the axes argument gives the
same axes and the refused ones stay refused; host arrays come back with the
elements a transform does not write left as they were (gaps, extents beyond the
result, an input inside the output's span) and dense outputs of any order whole,
also when the staging buffers still hold an earlier call's data."""
import numpy as np
import pytest

import rocket_fft_amd as R
from helpers import rel_l2


@pytest.mark.parametrize("axes", [[0, 2], np.array([0, 2]), np.array([0, 2], np.int32),
                                  np.array([0.0, 2.0]), (0, 2), np.array([0, 2], np.uint64),
                                  np.array([0, 9, 2])[::2], [np.int64(0), 2]])
def test_axes_forms(axes):
    S, keep = R._axes_struct(axes, 3)
    assert S.nitems == 2 and S.itemsize == 8 and list(S.shape_and_strides) == [2, 8]
    assert [int(v) for v in np.frombuffer(keep, np.uint64)] == [0, 2]


@pytest.mark.parametrize("axes,err", [([3], ValueError), ([-1], ValueError),
                                      (np.array([3]), ValueError), (np.array([-1]), ValueError),
                                      (np.array(1), TypeError), ([[0, 1]], TypeError)])
def test_axes_refused(axes, err):
    with pytest.raises(err):
        R._axes_struct(axes, 3)


def test_axes_empty():
    for axes in ([], np.array([], np.int64), np.array([])):
        S, _ = R._axes_struct(axes, 3)
        assert S.nitems == 0


def _crandn(rs, shape):
    return rs.standard_normal(shape) + 1j * rs.standard_normal(shape)


OUTS = {
    "c": lambda n: np.full((4, n), 7 + 0j),
    "f": lambda n: np.full((n, 4), 7 + 0j).T,
    "reversed": lambda n: np.full((4, n), 7 + 0j)[::-1, ::-1],
    "gaps": lambda n: np.full((4, 2 * n), 7 + 0j)[:, ::2],
    "rows": lambda n: np.full((8, n), 7 + 0j)[::2],
    "larger": lambda n: np.full((6, n + 3), 7 + 0j),
}


@pytest.mark.gpu
@pytest.mark.parametrize("layout", sorted(OUTS))
@pytest.mark.parametrize("n", [1, 30])
def test_host_output_layouts(layout, n):
    rs = np.random.RandomState(3)
    R.c2c(_crandn(rs, (64, 64)), np.empty((64, 64), complex), np.array([1]), True, 1.0)
    x = _crandn(rs, (4, n))
    out = OUTS[layout](n)
    whole = out if out.base is None else out.base
    R.c2c(x, out, np.array([1]), True, 1.0)
    assert rel_l2(out[:4, :n], np.fft.fft(x, axis=1)) <= 1e-13
    assert (whole == 7).sum() == whole.size - 4 * n  # the rest as it was
    r = rs.standard_normal((4, 2 * n))  # half spectrum into extents beyond n + 1
    half = np.full((5, n + 4), 7 + 0j)
    R.r2c(r, half, np.array([1]), True, 1.0)
    assert rel_l2(half[:4, :n + 1], np.fft.rfft(r, axis=1)) <= 1e-13
    assert (half == 7).sum() == half.size - 4 * (n + 1)


@pytest.mark.gpu
def test_host_input_inside_output():
    rs = np.random.RandomState(4)
    buf = np.zeros((4, 32), complex)
    x = _crandn(rs, (4, 32))
    buf[:] = x
    R.c2c(buf, buf, np.array([1]), True, 1.0)  # in place
    assert rel_l2(buf, np.fft.fft(x, axis=1)) <= 1e-13
    buf[:] = x
    R.c2c(buf[:2], buf[2:], np.array([1]), True, 1.0)  # next to each other
    assert rel_l2(buf[2:], np.fft.fft(x[:2], axis=1)) <= 1e-13
    assert np.array_equal(buf[:2], x[:2])
