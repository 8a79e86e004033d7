"""The dependency engine's resident tiles: grids whose 32 x 32 tiles all fit the
chip (no launch rounds before), grids that reach that point after some rounds
(every round tile shape), and more contexts at once than fit, whose tiles wait
for others not yet started and leave.  Bit-identical with the oracle, or with
the context stepped alone."""
import numpy as np
import pytest

from parallem_amd import lemhip, synth

pytestmark = pytest.mark.gpu

FIELDS = ["fd", "fa", "dem", "soilT", "stone", "fines", "depo"]
COUNTS = ["fa_uncomputed", "sed_uncomputed"]


def _dem(h, w, seed, frame):
    z = synth.fbm_surface(max(h, w, 3), np.random.default_rng(seed))[:h, :w].copy()
    synth.add_tilt(z)
    if frame:
        z[:1] = z[-1:] = synth.NODATA
        z[:, :1] = z[:, -1:] = synth.NODATA
    return z


def _against_oracle(z, flow, steps, tuning=None):
    from oracle import oracle as O
    h, w = z.shape
    rain = np.full(z.shape, 900.0)
    ctx = lemhip.LemContext(lemhip.default_params(w, h, flow), lemhip.FP64, 0)
    ctx.init_state(z, rain, soilT_mode="nonneg")
    if tuning:
        ctx.set_tuning(**tuning)
    orc = O.Oracle(z, rain, O.default_params(w, h, flow), soilT_mode="nonneg", openmp=True)
    for k in range(steps):
        ctx.step(-1000 + k)
        orc.step(-1000 + k)
        s = ctx.summary()
        for f in FIELDS:
            assert np.array_equal(ctx.download(f), orc[f], equal_nan=True), f"step {k}: {f}"
        for f in COUNTS:
            assert s[f] == orc.scalars()[f], f"step {k}: {f}"
    ctx.close()


# one cell, one tile with and without a second one beside or below it, cells on
# every tile edge and corner, a DEM without a nodata frame
@pytest.mark.parametrize("flow", [0, 1])
@pytest.mark.parametrize("frame,size", [(f, s) for f in (False, True) for s in
                                        ((1, 1), (3, 40), (32, 32), (33, 31), (31, 65), (64, 64), (97, 130))
                                        if not f or min(s) > 2])
def test_all_tiles_resident(size, flow, frame):
    _against_oracle(_dem(*size, seed=size[0] + flow, frame=frame), flow, steps=3)


# more tiles than the chip holds at once (at most 7 per compute unit): launch
# rounds in each tile shape first
@pytest.mark.parametrize("tile", [(64, 16), (32, 32), (128, 8)])
def test_resident_after_launch_rounds(tile):
    _against_oracle(_dem(1370, 1490, seed=5, frame=True), 0, steps=1, tuning=dict(dag_tile=tile, dag_batch=4))


def test_more_contexts_than_fit_at_once():
    """Three contexts of 900 to 1000 tiles each, stepped together: not all
    tiles of a context need be on the chip at the same time."""
    n = 3
    dems = [_dem(980 - 32 * k, 1010, seed=40 + k, frame=True) for k in range(n)]

    def make(k):
        h, w = dems[k].shape
        c = lemhip.LemContext(lemhip.default_params(w, h, k % 2), lemhip.FP64, 0)
        c.init_state(dems[k], np.full(dems[k].shape, 900.0), soilT_mode="nonneg")
        return c

    together = [make(k) for k in range(n)]
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
