"""Plateau fronts on a grid of more plateau tiles than compute units: eight
rounds per launch at first, sixteen once few tiles move, in both passes."""
import numpy as np
import pytest

from parallem_amd import lemhip

pytestmark = pytest.mark.gpu


def _flats(h, w):
    """A mesa drained through one notch (flat on the DEM itself: slope marks)
    above a basin that floods to one sill (flat on the raised surface)."""
    rng = np.random.default_rng(11)
    z = 300.0 + np.arange(h)[:, None] * 0.5 + rng.random((h, w))
    m = h // 2
    z[19:m - 19, 29:w - 29] = 901.0
    z[20:m - 20, 30:w - 30] = 900.0
    z[m // 2, 29] = 800.0
    z[m:h - 10, 20:w - 20] = 950.0
    z[m + 1:h - 11, 21:w - 21] = 700.0 + 10.0 * rng.random((h - 12 - m, w - 42))
    z[m + 40, w - 21] = 930.0
    z[0] = z[-1] = -9999.0
    z[:, 0] = z[:, -1] = -9999.0
    return z


@pytest.mark.parametrize("flow", [0, 1])
@pytest.mark.parametrize("choice", [4, 8, 16])
def test_fronts_across_many_tiles(flow, choice):
    from oracle import oracle as O
    h, w = 531, 790
    z, rain = _flats(h, w), np.full((h, w), 1000.0)
    ctx = lemhip.LemContext(lemhip.default_params(w, h, flow), lemhip.FP64, 0)
    ctx.init_state(z, rain, soilT_mode="nonneg")
    ctx.set_tuning(plateau_rounds_per_launch=choice)
    orc = O.Oracle(z, rain, O.default_params(w, h, flow), soilT_mode="nonneg", openmp=True)
    for k in range(2):
        ctx.step(-1000 + k)
        orc.step(-1000 + k)
        s, o = ctx.summary(), orc.scalars()
        for f in ("plateau_rounds1", "plateau_rounds2"):
            assert s[f] == o[f], f"step {k}: {f}"
        for f in ("fd", "SFD", "Slopes", "fa", "dem"):
            assert np.array_equal(ctx.download(f), orc[f], equal_nan=True), f"step {k}: {f}"
        if k == 0:
            assert s["plateau_rounds1"] > 500 and s["plateau_rounds2"] > 500
    ctx.close()
