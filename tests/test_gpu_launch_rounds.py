"""The dependency engine's launch rounds, which run only where more 32 x 32 tiles
are unfinished than the chip holds (at most 7 per compute unit)."""
import numpy as np
import pytest

from parallem_amd import lemhip, synth

pytestmark = pytest.mark.gpu


def _context(z, flow=0, precision=lemhip.FP64, **tuning):
    h, w = z.shape
    c = lemhip.LemContext(lemhip.default_params(w, h, flow), precision, 0)
    c.init_state(z, np.full(z.shape, 900.0), soilT_mode="nonneg")
    c.set_tuning(**tuning)
    return c


@pytest.mark.parametrize("precision", [lemhip.FP64, lemhip.FP32_KAHAN])
def test_autotune_keeps_choices_it_did_not_time(precision):
    """Where resident tiles take the whole pass, every tile shape and batch runs
    the same launches: the tuner leaves both as they were."""
    z = synth.fbm_512(side=200, seed_offset=34).z
    c = _context(z, 0, precision, dag_tile=(16, 64), dag_batch=7, fp32_tree_sediment=0)
    c.autotune()
    c.step(-1000)
    t = c.tuning()
    assert tuple(t["dag_tile"]) == (16, 64) and t["dag_batch"] == 7
    assert all(x > 0 for x in t["tuned_ms"][:6] + t["tuned_ms"][11:14])
    c.close()


def test_autotune_chooses_where_launch_rounds_run():
    z = synth.fbm_surface(1500, np.random.default_rng(6))
    synth.add_tilt(z)
    c = _context(z, 0, lemhip.FP64, dag_batch=7)
    c.autotune()
    c.step(-1000)
    assert c.tuning()["dag_batch"] in (4, 8, 16, 32)
    c.close()


FIELDS = ["fd", "fa", "dem", "soilT", "stone", "fines", "depo"]
COUNTS = ["fa_uncomputed", "sed_uncomputed"]
SHAPES = [(64, 16), (32, 32), (16, 64), (128, 8), (64, 32), (32, 64)]


def _relief(h, w, seed):
    z = synth.fbm_surface(max(h, w), np.random.default_rng(seed))[:h, :w].copy()
    synth.add_tilt(z)
    z[0] = z[-1] = synth.NODATA
    z[:, 0] = z[:, -1] = synth.NODATA
    return z


@pytest.fixture(scope="module", params=[0, 1])
def stepped_oracle(request):
    """2021 tiles: more than the chip holds."""
    from oracle import oracle as O
    flow, z = request.param, _relief(1370, 1490, seed=7)
    h, w = z.shape
    orc = O.Oracle(z, np.full(z.shape, 900.0), O.default_params(w, h, flow), soilT_mode="nonneg", openmp=True)
    orc.step(-1000)
    return flow, z, {f: np.array(orc[f]) for f in FIELDS}, dict(orc.scalars())


# 4 launches between host checks: resident tiles take over in the middle; 256:
# the rounds resolve (nearly) every cell
@pytest.mark.parametrize("batch", [4, 256])
@pytest.mark.parametrize("tile", SHAPES)
def test_every_shape_against_the_oracle(stepped_oracle, tile, batch):
    flow, z, fields, scalars = stepped_oracle
    c = _context(z, flow, dag_tile=tile, dag_batch=batch)
    c.profile(True)
    c.step(-1000)
    p = c.profile_read()
    assert p["fa_rounds"][1] >= batch and p["sed_rounds"][1] >= batch
    for f in FIELDS:
        assert np.array_equal(c.download(f), fields[f], equal_nan=True), f
    s = c.summary()
    for f in COUNTS:
        assert s[f] == scalars[f], f
    c.close()


@pytest.mark.parametrize("tile", SHAPES)
@pytest.mark.parametrize("flow", [0, 1])
def test_fp32_rounds_equal_resident_tiles(flow, tile):
    """FP32 form with both passes on the engine: a DEM alone, all of whose tiles are
    resident, and inside a nodata grid of 2209 tiles, whose launch rounds take
    nearly every cell: bit-identical."""
    h, w, y, x = 301, 411, 517, 709
    z = _relief(h, w, seed=8)
    big = np.full((1500, 1500), synth.NODATA)
    big[y:y + h, x:x + w] = z
    engine = dict(fp32_integer_fa=0, fp32_tree_sediment=0)
    alone = _context(z, flow, lemhip.FP32_KAHAN, **engine)
    rounds = _context(big, flow, lemhip.FP32_KAHAN, dag_tile=tile, dag_batch=256, **engine)
    rounds.profile(True)
    for k in range(2):
        alone.step(-1000 + k)
        rounds.step(-1000 + k)
        for f in FIELDS:
            part = rounds.download(f).reshape(1500, 1500)[y:y + h, x:x + w]
            assert np.array_equal(part, alone.download(f).reshape(h, w), equal_nan=True), f"step {k}: {f}"
        for f in COUNTS:
            assert rounds.summary()[f] == alone.summary()[f], f"step {k}: {f}"
    assert rounds.profile_read()["fa_rounds"][1] >= 256
    alone.close()
    rounds.close()


def test_fp32_contexts_that_do_not_fit_at_once():
    """Three FP32 contexts of some 950 tiles each, both direction types, stepped
    together: tiles wait for others that have not started, and leave."""
    dems = [_relief(980 - 32 * k, 1010, seed=50 + k) for k in range(3)]

    def make(k):
        return _context(dems[k], (k + 1) % 2, lemhip.FP32_KAHAN, fp32_integer_fa=0, fp32_tree_sediment=0)

    together = [make(k) for k in range(3)]
    for _ in range(2):
        lemhip.step_group(together)
    for k, c in enumerate(together):
        alone = make(k)
        alone.run(-1000, 2)
        for f in FIELDS:
            assert np.array_equal(c.download(f), alone.download(f), equal_nan=True), f"context {k}: {f}"
        alone.close()
    for c in together:
        c.close()


def test_time_of_looking_for_the_end_of_the_rounds():
    """8192^2: looking every 4 launches whether the unfinished tiles fit the chip costs
    little more than every 16 (3%; with a listing of the whole grid each time, 19%)."""
    z = synth.fbm_surface(2048, np.random.default_rng(9))
    z = np.block([[z, z[:, ::-1]], [z[::-1], z[::-1, ::-1]]])
    z = np.block([[z, z], [z, z]])
    synth.add_tilt(z)
    z[0] = z[-1] = synth.NODATA
    z[:, 0] = z[:, -1] = synth.NODATA
    c = _context(z, 0, dag_tile=(64, 16))
    c.flow_direction(-1000)
    c.runoff()
    ms = {}
    for batch in (16, 4) * 6:
        c.set_tuning(dag_batch=batch)
        c.profile(True)
        c.flow_accum(-1000)
        ms[batch] = min(ms.get(batch, 1e9), c.profile_read()["flow_accum"][0])
    c.close()
    assert 0 < ms[4] < 1.1 * ms[16], ms
