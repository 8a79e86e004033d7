"""Integer flow accumulation of the FP32 form at the edges of its 64 x 32 tiles:
one tile, one cell less and one more each way, whole and ragged rows of tiles;
the dependency engine is the other side, and the two agree to 1e-9 relative
(the engine's float pairs hold 48 bits, the integer sums are exact)."""
import numpy as np
import pytest

from parallem_amd import lemhip, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w, h", [(63, 31), (64, 32), (65, 33), (128, 96), (129, 65), (191, 300)])
def test_tile_edges(w, h):
    dem = synth.fbm_512(side=320, seed_offset=7)
    z = np.ascontiguousarray(dem.z[:h, :w])
    ctx = {}
    for integer in (1, 0):
        c = lemhip.LemContext(lemhip.default_params(w, h, 0, runiniter=0), lemhip.FP32_KAHAN, 0)
        c.init_state(z, np.ascontiguousarray(dem.rain[:h, :w]), soilT_mode="nonneg")
        c.set_tuning(fp32_integer_fa=integer)
        c.step(-1000)
        ctx[integer] = c
    m = ctx[1].download("mask") == 1
    assert np.array_equal(ctx[1].download("fd"), ctx[0].download("fd"))
    a, b = ctx[1].download("fa"), ctx[0].download("fa")
    assert float(np.max(np.abs(a[m] - b[m]) / np.maximum(b[m], 1e-30))) <= 1e-9
    assert np.array_equal(a[~m], b[~m])
    assert ctx[1].summary()["fa_uncomputed"] == ctx[0].summary()["fa_uncomputed"]
