"""16-bit column codes of a sliced ELL (tfs_layout_short_columns): every column
comes back, at the edges of a window and of their number, and in slices of odd,
even and no width; one window too many is refused."""
import numpy as np
import pytest

from tflows_amd import mesh


def check(widths, cols):
    off = 64 * np.concatenate(([0], np.cumsum(widths)))
    got = mesh.layout_short_columns(off, cols)
    return got is not None and np.array_equal(got, cols)


@pytest.mark.parametrize("widths", [[], [0], [1], [2], [7, 0, 6, 3], [9, 16]])
def test_widths(widths):
    u = np.random.default_rng(2)
    assert check(widths, u.integers(0, 3 * 4096, 64 * sum(widths)))


@pytest.mark.parametrize("last", [4095, 4096, 2**31 - 1])
def test_window_edges(last):
    cols = np.zeros(128, np.int64)
    cols[5], cols[127], cols[64] = last, 4096, last - 1
    assert check([2], cols)


@pytest.mark.parametrize("windows,ok", [(16, True), (17, False)])
def test_number_of_windows(windows, ok):
    cols = 4096 * (np.arange(192) % windows)
    assert check([3], cols) == ok
    assert check([0, 3, 1], np.concatenate((cols, np.zeros(64, int)))) == ok


def test_random_order_is_refused():
    assert mesh.layout_short_columns([0, 384], np.random.default_rng(3).integers(0, 10**6, 384)) \
        is None
