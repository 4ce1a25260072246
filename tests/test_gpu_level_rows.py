"""Synthesis levels in the register kernel against the general one (the
two-wave level shape) where blocks, segments and 4x4 groups end: sides around
multiples of 2, 4, 8 and 64 at every level, 5/3 and 9/7, int16 and int32 bands,
tiles of even origin, and tiles with odd origins and of a few pixels, which keep
their depth in the general kernel.  The same bytes, and under 5/3 the source."""
import numpy as np
import pytest

import signinum_amd as S

pytestmark = pytest.mark.gpu

ROWS, ROWS_SMALL, GENERAL = 1, 0, 3  # dwt shapes: 64x64 blocks by four waves (and 32x32), by two


def _decode(session, plan, shape, n):
    plan.dwt_shape = shape
    for s in plan.surfaces[:n]:
        s.fill(0x5A)
    plan.decode(S.MODE_GRAPH)
    session.synchronize()
    return [s.to_numpy() for s in plan.surfaces[:n]]


def _stream(rng, w, h, depth, reversible, **opts):
    img = rng.integers(0, 1 << depth, (h, w, 3), dtype=np.uint8 if depth == 8 else np.uint16)
    return img, S.encode_j2k_ht(img, bit_depth=depth, use_mct=0, reversible=reversible,
                                base_step=1 / 256, **opts)


@pytest.mark.parametrize("reversible", [1, 0])
@pytest.mark.parametrize("depth", [8, 16])
@pytest.mark.parametrize("w,h,levels,tiles", [
    (30, 370, 2, {}), (130, 270, 3, {}), (131, 269, 4, {}), (132, 268, 2, {}), (133, 267, 3, {}),
    (134, 266, 4, {}), (135, 265, 2, {}), (143, 257, 4, {}), (257, 143, 4, {}), (260, 140, 4, {}),
    (389, 40, 2, {}), (200, 100, 3, dict(tile_width=128, tile_height=64)),
    (405, 73, 2, dict(tile_width=64, tile_height=128))])
def test_equal_to_the_general_kernel(session, reversible, depth, w, h, levels, tiles):
    """One geometry a plan, every depth in the register kernel."""
    rng = np.random.default_rng(depth + w)
    img, cs = _stream(rng, w, h, depth, reversible, levels=levels, **tiles)
    fmt = S.PixelFormat.RGB8 if depth == 8 else S.PixelFormat.RGB16
    # more components than a level chain takes, so that each depth is a launch
    plan = S.TilePlan(session, [cs] * 172, fmt)
    got = {}
    for shape, kernel in ((ROWS, "rows"), (ROWS_SMALL, None), (GENERAL, "general")):
        plan.dwt_shape = shape
        ran = [k.split("-", 1)[1] for stage, k, _n in plan.kernels() if stage.startswith("levels")]
        assert len(ran) == levels - 1
        assert kernel is None or set(ran) == {kernel}
        got[shape] = _decode(session, plan, shape, 2)
    for shape in (ROWS, ROWS_SMALL):
        for a, b in zip(got[shape], got[GENERAL]):
            assert np.array_equal(a, b), shape
    if reversible:
        assert np.array_equal(got[ROWS][1], img)
    plan.close()


@pytest.mark.parametrize("reversible", [1, 0])
@pytest.mark.parametrize("depth", [8, 16])
def test_depths_with_other_tiles(session, reversible, depth):
    """Odd origins and sides under 8 beside the others: no depth in the register
    kernel where one of its levels does not fit it."""
    rng = np.random.default_rng(depth)
    streams, imgs = [], []
    for w in (30, 131, 135, 257, 389):
        img, cs = _stream(rng, w, 400 - w, depth, reversible, levels=2 + w % 3, tile_width=101,
                          tile_height=77)
        imgs.append(img)
        streams.append(cs)
    fmt = S.PixelFormat.RGB8 if depth == 8 else S.PixelFormat.RGB16
    plan = S.TilePlan(session, streams * 25, fmt)
    plan.dwt_shape = ROWS
    assert {k.split("-", 1)[1] for stage, k, _n in plan.kernels() if stage.startswith("levels")} == \
        {"general"}
    got = {shape: _decode(session, plan, shape, len(streams)) for shape in (ROWS, GENERAL)}
    for a, b, img in zip(got[ROWS], got[GENERAL], imgs):
        assert np.array_equal(a, b), img.shape
        assert not reversible or np.array_equal(a, img)
    plan.close()
