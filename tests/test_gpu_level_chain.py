"""Plans whose lowest levels go in one launch (few components) and plans past
that line: levels that differ between tiles, regions, reduced sizes, 5/3 and
9/7, replayed several times, against the source or the per-tile path."""
import numpy as np
import pytest

import signinum_amd as S
from signinum_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles,levels,size,chained", [
    (1, (5,), 70, 4), (3, (6, 3), 70, 2), (7, (2,), 70, 0), (4, (5, 5, 1), 70, 4), (171, (4,), 70, 0),
    (2, (3,), 80, 2), (24, (2, 4), 200, 0)])
@pytest.mark.parametrize("reversible", [1, 0])
def test_replays_equal_the_per_tile_path(session, tiles, levels, size, chained, reversible):
    rng = np.random.default_rng(tiles)
    imgs = [synth.tissue_rgb(rng, size + 20 + 13 * (k % 3), size + 5 * (k % 4)) for k in range(12)]
    streams = [S.encode_j2k_ht(imgs[k % 12], levels=levels[k % len(levels)], reversible=reversible,
                               use_mct=1) for k in range(tiles)]
    plan = S.TilePlan(session, streams, S.PixelFormat.RGB8)
    kernels = [k for stage, k, _n in plan.kernels() if stage.startswith("levels")]
    assert sum("chain" in k for k in kernels) == chained, kernels
    # levels of at least 8x8 lift in registers, also inside a chain
    assert size != 80 or set(kernels) == {("5/3" if reversible else "9/7") + "-chain-rows"}
    plan.decode(S.MODE_PLAIN)
    session.synchronize()
    want = [s.to_numpy() for s in plan.surfaces]
    if reversible:
        assert all(np.array_equal(w, imgs[k % 12]) for k, w in enumerate(want))
    for _ in range(3):
        for s in plan.surfaces:
            s.fill(0)
        plan.decode(S.MODE_GRAPH)
        session.synchronize()
        assert all(np.array_equal(s.to_numpy(), w) for s, w in zip(plan.surfaces, want))
    plan.close()


def test_regions_and_reduced_sizes(session):
    img = synth.texture_rgb(np.random.default_rng(2), 700, 500)
    d = S.J2kDecoder(S.encode_j2k_lossless(img, levels=6), session)
    for roi in ((0, 0, 64, 64), (333, 77, 130, 200), (650, 450, 50, 50)):
        x, y, w, h = roi
        got = d.decode_region_to_numpy(S.PixelFormat.RGB8, roi)
        assert np.array_equal(got, img[y:y + h, x:x + w])
