"""The 16-bit final stage of 8-bit RGB tiles where its blocks, chunks and
4x4 groups end: widths and heights around multiples of 4, 8 and 64, one
level and several, padded and unaligned surfaces, tiles that it leaves to the
general kernel beside tiles that it takes, against the source pixels."""
import numpy as np
import pytest

import signinum_amd as S
from signinum_amd import synth

pytestmark = pytest.mark.gpu


class _Surface:
    """A tile inside a larger device image: any offset and pitch."""

    def __init__(self, base, offset, pitch, height):
        self.device_ptr = base.device_ptr + offset
        self.pitch_bytes = pitch
        self.byte_len = pitch * height


@pytest.mark.parametrize("w", [8, 9, 63, 64, 65, 66, 67, 71, 128, 130, 131, 197])
@pytest.mark.parametrize("h,levels", [(8, 1), (9, 2), (64, 1), (65, 5), (66, 3), (67, 2), (131, 4)])
def test_sizes(session, w, h, levels):
    img = np.random.default_rng(w * 7 + h).integers(0, 256, (h, w, 3), dtype=np.uint8)
    cs = S.encode_j2k_lossless(img, levels=levels)
    plan = S.TilePlan(session, [cs], S.PixelFormat.RGB8)
    assert [k for stage, k, _n in plan.kernels() if stage == "final"] == ["5/3-rgb8"]
    for mode in (S.MODE_GRAPH, S.MODE_PLAIN):
        plan.surfaces[0].fill(0x5A)
        plan.decode(mode)
        session.synchronize()
        assert np.array_equal(plan.surfaces[0].to_numpy(), img)
    plan.close()


@pytest.mark.parametrize("offset,pitch_extra", [(0, 0), (4, 8), (1, 0), (3, 5), (0, 2)])
def test_offsets_pitches_and_neighbouring_kernels(session, offset, pitch_extra):
    """Tiles of both kernels in one plan (RGB8 beside RGBA8, Gray8, tiles too
    small and multi-tile images with odd tile origins), written into images of
    any alignment; bytes outside the tiles stay."""
    rng = np.random.default_rng(11)
    shapes = [(70, 66, S.PixelFormat.RGB8, {}), (5, 9, S.PixelFormat.RGB8, {}),
              (90, 70, S.PixelFormat.RGBA8, {}), (64, 64, S.PixelFormat.RGB8, {}),
              (150, 140, S.PixelFormat.RGB8, dict(tile_width=51, tile_height=53)),
              (77, 40, S.PixelFormat.GRAY8, {})]
    imgs, streams, surfs, bases = [], [], [], []
    for w, h, fmt, opts in shapes:
        ch = 1 if fmt == S.PixelFormat.GRAY8 else 3
        img = rng.integers(0, 256, (h, w, ch), dtype=np.uint8)
        imgs.append(img)
        streams.append(S.encode_j2k_ht(img, levels=3, use_mct=1 if ch == 3 else 0, **opts))
        pitch = w * fmt.bytes_per_pixel + pitch_extra
        base = S.DeviceSurface(session, pitch * h + 16, 1, S.PixelFormat.GRAY8)
        base.fill(0xC3)
        bases.append(base)
        surfs.append(_Surface(base, offset, pitch, h))
    plan = S.TilePlan(session, streams, [s[2] for s in shapes], surfaces=surfs)
    assert [k for stage, k, _n in plan.kernels() if stage == "final"] == ["5/3-rgb8", "5/3-general"]
    plan.decode(S.MODE_GRAPH)
    session.synchronize()
    for (w, h, fmt, _o), img, base in zip(shapes, imgs, bases):
        raw = base.to_numpy().reshape(-1)
        bpp = fmt.bytes_per_pixel
        pitch = w * bpp + pitch_extra
        rows = raw[offset:offset + pitch * h].reshape(h, pitch)
        got = rows[:, :w * bpp].reshape(h, w, bpp)
        assert np.array_equal(got[..., :img.shape[2]], img), (w, h, fmt)
        assert (rows[:, w * bpp:] == 0xC3).all() and (raw[:offset] == 0xC3).all()
        assert (raw[offset + pitch * h:] == 0xC3).all()
    plan.close()
