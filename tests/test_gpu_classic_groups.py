"""Classic code-blocks where the kernel's groups, stripes and shapes end: sides
around eight columns and four rows, blocks of both kernel sizes, every style
with and without raw segments, each lane count, more blocks than the first
lanes take, and damaged bytes (0xFF runs: markers and stuffing anywhere),
against the oracle."""
import numpy as np
import pytest

import signinum_amd as S
from signinum_amd import synth
from tests import oracle_ref as O

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 2, 2), (7, 3, 3, 2), (8, 4, 3, 2), (9, 5, 4, 3), (97, 75, 6, 6), (130, 9, 8, 2),
          (5, 90, 2, 8), (260, 4, 10, 2), (3, 300, 2, 10), (64, 64, 6, 6)]


@pytest.mark.parametrize("lanes", ["16", "4", "3", "2", "1", "32", "r32", "r16"])
@pytest.mark.parametrize("style", [0, 1, 2 | 4, 8, 1 | 2 | 4 | 8 | 0x20])
def test_blocks_of_every_shape(session, oracle, monkeypatch, style, lanes):
    monkeypatch.setenv("SGN_CLASSIC_LANES", lanes)
    rng = np.random.default_rng(style)
    good, bad = [], []
    for w, h, cbw, cbh in SHAPES:
        for img in (rng.integers(0, 256, (h, w, 3), dtype=np.uint8), synth.tissue_rgb(rng, w, h)):
            cs = S.encode_j2k_classic(img, cb_style=style, cb_width_log2=cbw, cb_height_log2=cbh,
                                      levels=2, use_mct=1)
            good.append((cs, img))
            data = bytearray(cs)
            start = data.index(b"\xff\x93") + 60
            if len(data) - start > 100:
                at, n = int(rng.integers(start, len(data) - 50)), int(rng.integers(1, 20))
                data[at:at + n] = b"\xff" * n if w % 2 else rng.bytes(n)
                if O.decode_rc(bytes(data), 1) == 0:
                    bad.append((bytes(data), O.decode(bytes(data), 1)))
    for cases in (good, bad):
        plan = S.TilePlan(session, [c for c, _ in cases], S.PixelFormat.RGB8)
        for mode in (S.MODE_GRAPH, S.MODE_GRAPH, S.MODE_PLAIN):
            for s in plan.surfaces:
                s.fill(0x5A)
            plan.decode(mode)
            session.synchronize()
            for (cs, want), s in zip(cases, plan.surfaces):
                assert np.array_equal(s.to_numpy(), want), (want.shape, mode)
        plan.close()


def test_more_blocks_than_lanes(session, oracle):
    """3072 blocks of 4x4 to 16x16: lanes end and take the next ones while the
    others of their wave are in the middle of theirs."""
    rng = np.random.default_rng(3)
    imgs = [rng.integers(0, 256, (128, 128, 3), dtype=np.uint8) if k % 3 else
            synth.near_white_rgb(rng, 128, 128) for k in range(16)]
    streams = [S.encode_j2k_classic(v, cb_width_log2=2 + k % 3, cb_height_log2=2 + k % 2, levels=1)
               for k, v in enumerate(imgs)]
    plan = S.TilePlan(session, streams, S.PixelFormat.RGB8)
    for _ in range(3):
        for s in plan.surfaces:
            s.fill(0)
        plan.decode(S.MODE_GRAPH)
        session.synchronize()
        assert all(np.array_equal(s.to_numpy(), v) for s, v in zip(plan.surfaces, imgs))
    plan.close()
