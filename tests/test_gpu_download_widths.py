"""Downloads widened on the host: every element width on both sides of the size up
to which they are packed straight into pinned memory (8 MB as the host holds
them, 4 MB packed), and what narrow fields gain by crossing the link narrow."""
import time

import numpy as np
import pytest

from parallem_amd import lemhip

pytestmark = pytest.mark.gpu


def _context(w, h, prec):
    c = lemhip.LemContext(lemhip.default_params(w, h, 0), prec, 0)
    c.init_state(np.full((h, w), 50.0))
    return c


@pytest.mark.parametrize("prec", [lemhip.FP64, lemhip.FP32_KAHAN])
@pytest.mark.parametrize("side", [1024, 1025, 1448, 1449])
def test_both_sides_of_the_border(side, prec):
    n = side * side
    rng = np.random.default_rng(side)
    c = _context(side, side, prec)
    mask = (rng.random(n) < 0.8).astype(np.int32)
    fd = rng.integers(0, 256, n).astype(np.int32)
    stone = rng.normal(0.0, 1e3, n).astype(np.float32).astype(np.float64)
    for f, v in (("mask", mask), ("fd", fd), ("stone", stone)):
        c.upload(f, v)
    assert np.array_equal(c.download("mask"), mask)
    assert np.array_equal(c.download("fd"), np.where(mask != 0, fd, -9999))
    assert np.array_equal(c.download("stone"), stone)
    c.close()


def test_time_of_narrow_fields():
    """The mask crosses the link in one byte a cell, directions in two: 0.08 and 0.13 ms
    on 1024^2, 0.22 each where both crossed it in four."""
    c = _context(1024, 1024, lemhip.FP64)
    c.upload("mask", np.ones(1024 * 1024, np.int32))
    ms = {"mask": 1e9, "fd": 1e9}
    for _ in range(30):
        for f in ms:
            t = time.perf_counter()
            c.download(f)
            ms[f] = min(ms[f], time.perf_counter() - t)
    c.close()
    assert ms["mask"] < 0.85 * ms["fd"], ms
