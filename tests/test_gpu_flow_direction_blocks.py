"""Flow directions with one and with four 16-row tiles per block (grids below
and above two four-tile blocks per compute unit), ragged on both axes; directions,
slopes and plateau rounds are the oracle's."""
import numpy as np
import pytest

from parallem_amd import lemhip, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h, w", [(15, 65), (113, 64), (1313, 1729)])
def test_against_oracle(h, w):
    from oracle import oracle as O
    z = synth.fbm_surface(max(h, w), np.random.default_rng(5))[:h, :w].copy() + 50.0
    z[h // 3:h // 3 + 9, w // 4:w // 4 + 20] = z[h // 3, w // 4]   # a flat
    z[0] = z[-1] = synth.NODATA
    z[:, 0] = z[:, -1] = synth.NODATA
    rain = np.full(z.shape, 900.0)
    ctx = lemhip.LemContext(lemhip.default_params(w, h, 1), lemhip.FP64, 0)
    ctx.init_state(z, rain, soilT_mode="nonneg")
    orc = O.Oracle(z, rain, O.default_params(w, h, 1), soilT_mode="nonneg", openmp=True)
    ctx.step(-1000)
    orc.step(-1000)
    s, o = ctx.summary(), orc.scalars()
    for f in ("sinkcount", "plateau_rounds1", "plateau_rounds2"):
        assert s[f] == o[f], f
    for f in ("fd", "SFD"):
        assert np.array_equal(ctx.download(f), np.where(orc["mask"] != 0, orc[f], -9999)), f
    assert np.array_equal(ctx.download("Slopes"), orc["Slopes"], equal_nan=True)
    ctx.close()
