"""Tiles that start at an odd row and an even column: the first row's halo left
of every block but the first in a row, which 5/3 and 9/7 read only there."""
import numpy as np
import pytest

import signinum_amd as S
from tests import oracle_ref as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,tw,th", [(257, 143, 101, 77), (101, 154, 101, 77), (140, 131, 140, 67)])
@pytest.mark.parametrize("reversible", [1, 0])
@pytest.mark.parametrize("levels", [1, 3])
def test_first_row_of_every_block(session, oracle, w, h, tw, th, reversible, levels):
    img = np.random.default_rng(w).integers(0, 256, (h, w, 3), dtype=np.uint8)
    cs = S.encode_j2k_ht(img, levels=levels, use_mct=1, reversible=reversible, base_step=1 / 64,
                         tile_width=tw, tile_height=th)
    want = O.decode(cs, 1).astype(int)
    plan = S.TilePlan(session, [cs], S.PixelFormat.RGB8)
    for mode in (S.MODE_GRAPH, S.MODE_PLAIN):
        plan.surfaces[0].fill(0x5A)
        plan.decode(mode)
        session.synchronize()
        d = np.abs(plan.surfaces[0].to_numpy().astype(int) - want).max()
        assert d <= (0 if reversible else 1), (mode, d)
    plan.close()


@pytest.mark.parametrize("shape", range(4))
def test_odd_columns_in_every_level_shape(session, oracle, shape):
    """9/7 levels with an odd x origin (loaded sample by sample): each row's
    band step, past the 32nd row of a thread too."""
    img = np.random.default_rng(6).integers(0, 256, (257, 143), dtype=np.uint8)
    cs = S.encode_j2k_ht(img, levels=2, use_mct=0, reversible=0, base_step=1 / 256, tile_width=101,
                         tile_height=77)
    want = O.decode(cs, int(S.PixelFormat.GRAY8)).astype(int)
    plan = S.TilePlan(session, [cs], S.PixelFormat.GRAY8)
    plan.dwt_shape = shape
    plan.surfaces[0].fill(0x5A)
    plan.decode(S.MODE_GRAPH)
    session.synchronize()
    assert np.abs(plan.surfaces[0].to_numpy().astype(int) - want).max() <= 1
    plan.close()
