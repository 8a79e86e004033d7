"""Downloads of every kind of field: packed on the device from a DEM's rectangle
(any width, any place in an atlas), widened to the host types, straight into
pinned memory up to 4 MB and in 2 MB chunks on several threads above."""
import numpy as np
import pytest

from parallem_amd import lemhip

pytestmark = pytest.mark.gpu

# (width, height): one cell, odd rows, a whole number of chunks, one value past
# the 4 MB border of an f64 field, several chunks with a remainder
SIZES = [(1, 1), (7, 3), (97, 64), (512, 1024), (713, 736), (1201, 907)]


def _values(rng, name, n):
    if name == "mask":
        return (rng.random(n) < 0.8).astype(np.int32)
    if name in lemhip.INT_FIELDS:
        return rng.integers(0, 256, n).astype(np.int32)
    return rng.normal(0.0, 1e3, 8 * n if name == "Slopes" else n)


def _expected(name, v, mask, prec):
    if name in ("fd", "SFD"):
        return np.where(mask != 0, v, -9999)
    if name in lemhip.INT_FIELDS or prec == lemhip.FP64 or name in ("dem", "soilT"):
        return v
    if name == "fa":            # float pair
        hi = v.astype(np.float32)
        return hi.astype(np.float64) + (v - hi).astype(np.float32).astype(np.float64)
    return v.astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("prec", [lemhip.FP64, lemhip.FP32_KAHAN])
@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("atlas", [False, True])
def test_download_returns_what_was_uploaded(size, prec, atlas):
    w, h = size
    n = w * h
    rng = np.random.default_rng(w * 1000 + h)
    z = rng.uniform(1.0, 100.0, n)
    if atlas:     # behind another DEM, so the rectangle starts at column 64
        W = lemhip.atlas_span([40, w])
        ctx = lemhip.LemAtlas(lemhip.default_params(W, h + 1, 0), W, h + 1, prec, 0)
        first = ctx.add(np.ones((h, 40)))
        assert first is not None
        slot = ctx.add(z.reshape(h, w))
        assert slot is not None
        up, down = (lambda f, v: ctx.upload(slot, f, v)), (lambda f: ctx.download(slot, f))
    else:
        ctx = lemhip.LemContext(lemhip.default_params(w, h, 0), prec, 0)
        ctx.init_state(z)
        up, down = ctx.upload, ctx.download
    mask = _values(rng, "mask", n)
    up("mask", mask)
    sent = {"mask": mask}
    for f in ("dem", "soilT", "stone", "fa", "fd", "SFD", "Slopes"):
        sent[f] = _values(rng, f, n)
        up(f, sent[f])
    for f, v in sent.items():
        assert np.array_equal(down(f), _expected(f, v, mask, prec)), f
    ctx.close()
