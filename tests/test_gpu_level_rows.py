"""Synthesis levels in the register kernel against the general one (the
two-wave level shape) where blocks, segments and 4x4 groups end: sides around
multiples of 2, 4, 8 and 64 at every level, 5/3 and 9/7, int16 and int32 bands,
tiles with odd origins and of a few pixels beside them.  The same bytes."""
import numpy as np
import pytest

import signinum_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("reversible", [1, 0])
@pytest.mark.parametrize("depth", [8, 16])
@pytest.mark.parametrize("tiled", [False, True])
def test_equal_to_the_general_kernel(session, reversible, depth, tiled):
    rng = np.random.default_rng(depth)
    dt = np.uint8 if depth == 8 else np.uint16
    streams = []
    for w in (30, 130, 131, 132, 133, 134, 135, 143, 257, 260, 389):
        h = 400 - w
        img = rng.integers(0, 1 << depth, (h, w), dtype=dt)
        opts = dict(tile_width=101, tile_height=77) if tiled else {}
        streams.append(S.encode_j2k_ht(img, bit_depth=depth, levels=2 + w % 3, use_mct=0,
                                       reversible=reversible, base_step=1 / 256, **opts))
    fmt = S.PixelFormat.GRAY8 if depth == 8 else S.PixelFormat.GRAY16
    # more components than a level chain takes, so that each depth is a launch
    plan = S.TilePlan(session, streams * 50, fmt)
    got = {}
    for shape in (0, 2):
        plan.dwt_shape = shape
        for s in plan.surfaces:
            s.fill(0x5A)
        plan.decode(S.MODE_GRAPH)
        session.synchronize()
        got[shape] = [s.to_numpy() for s in plan.surfaces[:len(streams)]]
    for a, b in zip(got[0], got[2]):
        assert np.array_equal(a, b), a.shape
    plan.close()
