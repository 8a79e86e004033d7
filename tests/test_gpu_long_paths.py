"""Depression routing where paths are longer than the walks that follow them:
basins that join along one path, and watershed pointers along a winding valley.
Bit-identical with the oracle."""
import numpy as np
import pytest

from parallem_amd import lemhip, synth

pytestmark = pytest.mark.gpu


def _falling_sills(h, w, outlet):
    """A channel of pits winding through every second row, its sills falling one
    after the other: every basin, and label 0 before them all, joins the next one
    along it.  outlet: a valid cell on the DEM's edge beside the first pit."""
    z = np.full((h, w), 1e7)
    n = w - 4
    for k, r in enumerate(range(2, h - 2, 2)):
        p = k * (n + 1) + np.arange(n + 1)
        v = 4e6 - p - 3.0 * (p % 2)
        z[r, 2:w - 2] = v[:n] if k % 2 == 0 else v[n - 1::-1]
        if r + 2 < h - 2:
            z[r + 1, w - 3 if k % 2 == 0 else 2] = v[n]
    z[0] = z[-1] = synth.NODATA
    z[:, 0] = z[:, -1] = synth.NODATA
    if outlet:
        z[1, 2], z[0, 2] = 4e6, 4e6 - 10
    return z


def _winding_valley(h, w, rough_rows=0, upwards=False):
    """A valley winding through every second row, falling all the way to a pit;
    the last rough_rows rows full of small basins instead."""
    z = np.full((h, w), 2000.0)
    n = w - 4
    for k, r in enumerate(range(2, h - 2 - rough_rows, 2)):
        fall = 1500.0 - 1e-4 * (k * (n + 1) + np.arange(n + 1))
        z[r, 2:w - 2] = fall[:n] if k % 2 == 0 else fall[n - 1::-1]
        if r + 2 < h - 2 - rough_rows:
            z[r + 1, w - 3 if k % 2 == 0 else 2] = fall[n]
    if rough_rows:
        z[h - rough_rows:] = 2000.0 + 50.0 * np.random.default_rng(1).random((rough_rows, w))
    z = np.ascontiguousarray(z[::-1]) if upwards else z
    z[0] = z[-1] = synth.NODATA
    z[:, 0] = z[:, -1] = synth.NODATA
    return z


def _equals_oracle(z, flow):
    from oracle import oracle as O
    h, w = z.shape
    rain = np.full(z.shape, 800.0)
    ctx = lemhip.LemContext(lemhip.default_params(w, h, flow), lemhip.FP64, 0)
    ctx.init_state(z, rain, soilT_mode="nonneg")
    orc = O.Oracle(z, rain, O.default_params(w, h, flow), soilT_mode="nonneg", openmp=True)
    ctx.step(-1000)
    orc.step(-1000)
    s, o = ctx.summary(), orc.scalars()
    for f in ("sinkcount", "plateau_rounds1", "plateau_rounds2"):
        assert s[f] == o[f], f
    for f in ("fd", "SFD"):   # downloads carry -9999 on nodata
        assert np.array_equal(ctx.download(f), np.where(orc["mask"] != 0, orc[f], -9999)), f
    assert np.array_equal(ctx.download("fa"), orc["fa"], equal_nan=True)
    ctx.close()


# 1307 and 2997 basins: more than a walk follows; 1103026: more than 2^20
@pytest.mark.parametrize("h, w, outlet, flow", [(40, 150, True, 0), (40, 150, True, 1), (7, 3000, True, 0),
                                                (2105, 2104, False, 0)])
def test_basins_joining_along_one_path(h, w, outlet, flow):
    _equals_oracle(_falling_sills(h, w, outlet), flow)


# few basins (three jumps before the walks), some 600 (two) and many (one)
@pytest.mark.parametrize("rough_rows", [0, 6, 100])
@pytest.mark.parametrize("upwards", [False, True])
def test_winding_valley(rough_rows, upwards):
    _equals_oracle(_winding_valley(1100, 1203, rough_rows, upwards), 0)


def test_time_of_a_winding_valley():
    """Depression routing of a valley of 8 million cells takes about 3 ms; walks
    to the valley's end, link by link, 89."""
    z = _winding_valley(4096, 4096)
    ctx = lemhip.LemContext(lemhip.default_params(4096, 4096), lemhip.FP32_KAHAN, 0)
    ctx.init_state(z, np.full(z.shape, 800.0), soilT_mode="nonneg")
    ctx.flow_direction(-1000)
    ctx.profile(True)
    ctx.flow_direction(-999)
    ms = ctx.profile_read()["depression"][0]
    ctx.close()
    assert 0 < ms < 30


def test_cut_off_basins_are_timed_as_depression_routing():
    """A row of basins inside a NaN ring: their spill heights take hundreds of
    relaxation passes, found necessary only once the surface was raised."""
    z = np.full((11, 800), 5000.0)
    c = np.arange(3, 797)
    z[5, 3:-3] = 500.0 + c + np.where(c % 2 == 0, 0.0, -3.0)
    z[1:-1, 1] = z[1:-1, -2] = z[1, 1:-1] = z[-2, 1:-1] = np.nan
    z[0] = z[-1] = synth.NODATA
    z[:, 0] = z[:, -1] = synth.NODATA
    ctx = lemhip.LemContext(lemhip.default_params(800, 11), lemhip.FP64, 0)
    ctx.init_state(z, np.full(z.shape, 800.0), soilT_mode="nonneg")
    ctx.flow_direction(-1000)
    ctx.profile(True)
    ctx.flow_direction(-999)
    p = ctx.profile_read()
    ctx.close()
    # hundreds of passes at some 10 us each, against a millisecond of other phases
    assert p["depression"][0] > 0.5 * p["fd"][0]
    assert p["depression"][1] == 1
