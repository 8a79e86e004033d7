"""Depression routing: basins that NaN heights cut off from the border (found
only after the surface was raised once), watershed pointers as long as a
serpentine valley, and a row of basins that join in one long path.
Bit-identical with the oracle."""
import numpy as np
import pytest

from parallem_amd import lemhip, synth

pytestmark = pytest.mark.gpu


def _nan_ring(h, w):
    rng = np.random.default_rng(3)
    z = synth.fbm_surface(max(h, w), rng)[:h, :w].copy() + 50.0
    z[20:50, 15:60] -= 30.0
    for r0, r1, c0, c1 in ((18, 52, 13, 62), (25, 45, 25, 50)):    # one ring inside another
        z[r0:r1, c0] = z[r0:r1, c1 - 1] = np.nan
        z[r0, c0:c1] = z[r1 - 1, c0:c1] = np.nan
    z[0] = z[-1] = synth.NODATA
    z[:, 0] = z[:, -1] = synth.NODATA
    return z


def _serpentine(h, w):
    """A valley winding through every second row, falling all the way to a pit."""
    z = np.full((h, w), 2000.0)
    height = 1500.0
    for k, r in enumerate(range(2, h - 2, 2)):
        cols = range(2, w - 2) if k % 2 == 0 else range(w - 3, 1, -1)
        for c in cols:
            z[r, c] = height
            height -= 0.05
        last = w - 3 if k % 2 == 0 else 2
        if r + 2 < h - 2:
            z[r + 1, last] = height
            height -= 0.05
    z[0] = z[-1] = synth.NODATA
    z[:, 0] = z[:, -1] = synth.NODATA
    return z


def _stairs(h, w):
    """A channel of pits whose sills rise one after the other: every basin's lowest
    sill is the last one's, so all of them join along one path."""
    z = np.full((h, w), 5000.0)
    c = np.arange(1, w - 1)
    z[h // 2, 1:-1] = 500.0 + c + np.where(c % 2 == 0, 0.0, -3.0)
    z[0] = z[-1] = synth.NODATA
    z[:, 0] = z[:, -1] = synth.NODATA
    return z


@pytest.mark.parametrize("flow", [0, 1])
@pytest.mark.parametrize("case", ["nan_ring", "serpentine", "stairs"])
def test_against_oracle(case, flow):
    from oracle import oracle as O
    z = {"nan_ring": lambda: _nan_ring(70, 90), "serpentine": lambda: _serpentine(131, 140),
         "stairs": lambda: _stairs(7, 1500)}[case]()
    h, w = z.shape
    rain = np.full(z.shape, 800.0)
    ctx = lemhip.LemContext(lemhip.default_params(w, h, flow), lemhip.FP64, 0)
    ctx.init_state(z, rain, soilT_mode="nonneg")
    orc = O.Oracle(z, rain, O.default_params(w, h, flow), soilT_mode="nonneg")
    for k in range(2):
        ctx.step(-1000 + k)
        orc.step(-1000 + k)
        s, o = ctx.summary(), orc.scalars()
        for f in ("sinkcount", "plateau_rounds1", "plateau_rounds2"):
            assert s[f] == o[f], f"step {k}: {f}"
        for f in ("fd", "SFD"):   # downloads carry -9999 on nodata, the outlet's cell among them when it is none
            assert np.array_equal(ctx.download(f), np.where(orc["mask"] != 0, orc[f], -9999)), f"step {k}: {f}"
        for f in ("fa", "dem", "soilT"):
            assert np.array_equal(ctx.download(f), orc[f], equal_nan=True), f"step {k}: {f}"
    ctx.close()


@pytest.mark.parametrize("h, w", [(15, 63), (16, 64), (17, 65), (33, 129), (64, 130)])
def test_basin_pairs_at_block_edges(h, w):
    """Many small basins with equal heights between them and holes in the mask,
    on grids one cell around whole 64 x 16 blocks."""
    from oracle import oracle as O
    rng = np.random.default_rng(h * 1000 + w)
    z = 100.0 + rng.integers(0, 6, (h, w)).astype(np.float64)
    z[rng.random((h, w)) < 0.03] = synth.NODATA
    rain = np.full(z.shape, 800.0)
    ctx = lemhip.LemContext(lemhip.default_params(w, h, 0), lemhip.FP64, 0)
    ctx.init_state(z, rain, soilT_mode="nonneg")
    orc = O.Oracle(z, rain, O.default_params(w, h, 0), soilT_mode="nonneg")
    ctx.step(-1000)
    orc.step(-1000)
    s, o = ctx.summary(), orc.scalars()
    for f in ("sinkcount", "nedges", "plateau_rounds1", "plateau_rounds2"):
        if f in s and f in o:
            assert s[f] == o[f], f
    for f in ("fd", "SFD"):
        assert np.array_equal(ctx.download(f), np.where(orc["mask"] != 0, orc[f], -9999)), f
    for f in ("fa", "dem"):
        assert np.array_equal(ctx.download(f), orc[f], equal_nan=True), f
    ctx.close()
