"""FP32 sediment contraction from both kinds of rounds: with one engine round a
1900^2 DEM leaves more open cells than the short-list bound, with three fewer;
the same cells compute as with the engine to the end, deposition and soil
thickness are bit-identical and stone within 1e-6 relative (a few float ulps
where a composed chain reached a cell), the form's own bound."""
import numpy as np
import pytest

from parallem_amd import lemhip, synth

pytestmark = pytest.mark.gpu

SHORT = 262144


def _step(dem, rounds):
    h, w = dem.z.shape
    c = lemhip.LemContext(lemhip.default_params(w, h, 0), lemhip.FP32_KAHAN, 0)
    c.init_state(dem.z, dem.rain, soilT_mode="nonneg")
    c.set_tuning(fp32_tree_sediment=rounds)
    c.step(-1000)
    out = {f: c.download(f) for f in ("depo", "soilT", "dem", "stone", "mask")}
    s = c.summary()
    c.close()
    return out, s


def test_short_and_long_lists():
    dem = synth.fbm_4096(side=1900)
    ref, s0 = _step(dem, 0)
    m = ref["mask"] == 1
    for rounds, long_list in ((1, True), (3, False)):
        got, s = _step(dem, rounds)
        assert (s["sed_open"] > SHORT) == long_list
        assert s["sed_uncomputed"] == s0["sed_uncomputed"]
        for f in ("depo", "soilT"):
            assert np.array_equal(got[f], ref[f]), f
        a, b = got["stone"][m], ref["stone"][m]
        assert float(np.max(np.abs(a - b) / np.abs(b))) <= 1e-6
