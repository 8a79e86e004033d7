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
