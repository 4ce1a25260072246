"""The register final stage of 8-bit RGB tiles under 9/7 and ICT where its
blocks, segments and 4x4 groups end, padded and unaligned surfaces: the same
bytes as the general kernel, which decodes the same tiles to RGBA8, and within
one grey level of the oracle; and the tiles that it leaves to that kernel (one
level, int32 band samples, odd origins, small sides)."""
import numpy as np
import pytest

import signinum_amd as S
from tests import oracle_ref as O

pytestmark = pytest.mark.gpu


def _encode(img, **opts):
    return S.encode_j2k_ht(img, reversible=0, use_mct=1, **opts)


def _finals(plan):
    return [k for stage, k, _n in plan.kernels() if stage == "final"]


def _check(session, streams, imgs, kernels):
    got = S.TilePlan(session, streams, S.PixelFormat.RGB8)
    ref = S.TilePlan(session, streams, S.PixelFormat.RGBA8)
    assert _finals(got) == kernels and _finals(ref) == ["9/7-general"]
    for mode in (S.MODE_GRAPH, S.MODE_PLAIN):
        for p in (got, ref):
            for s in p.surfaces:
                s.fill(0x5A)
            p.decode(mode)
        session.synchronize()
        for cs, img, a, b in zip(streams, imgs, got.surfaces, ref.surfaces):
            pix = a.to_numpy()
            assert np.array_equal(pix, b.to_numpy()[..., :3]), img.shape
            d = np.abs(pix.astype(int) - O.decode(cs, 1).astype(int)).max()
            assert d <= 1, (img.shape, d)
    got.close()
    ref.close()


@pytest.mark.parametrize("w", [8, 9, 10, 11, 63, 64, 65, 66, 67, 68, 69, 72, 130, 197])
@pytest.mark.parametrize("step,levels,kernel", [
    (1 / 16, (2, 3, 4), "9/7-rgb8"),
    (1 / 16, (1,), "9/7-general"),          # int16 low-pass samples, not f32
    (1 / 2048, (1, 2, 3), "9/7-general")])  # int32 band samples
def test_sizes(session, oracle, w, step, levels, kernel):
    rng = np.random.default_rng(w)
    imgs = [rng.integers(0, 256, (h, w, 3), dtype=np.uint8) for h in (8, 9, 64, 65, 66, 67, 68, 69, 131)]
    streams = [_encode(v, levels=levels[k % len(levels)], base_step=step) for k, v in enumerate(imgs)]
    _check(session, streams, imgs, [kernel])


def test_tiles_that_the_general_kernel_keeps(session, oracle):
    """Multi-tile images with odd tile origins and tiles too small, beside
    tiles of the register kernel."""
    rng = np.random.default_rng(4)
    imgs = [rng.integers(0, 256, s, dtype=np.uint8)
            for s in ((70, 66, 3), (5, 9, 3), (140, 150, 3), (64, 7, 3), (64, 64, 3))]
    streams = [_encode(v, levels=3, **(dict(tile_width=51, tile_height=53) if v.shape[0] == 140 else {}))
               for v in imgs]
    _check(session, streams, imgs, ["9/7-rgb8", "9/7-general"])


@pytest.mark.parametrize("offset,pitch_extra", [(4, 8), (1, 0), (3, 5), (0, 2)])
def test_offsets_and_pitches(session, offset, pitch_extra):
    rng = np.random.default_rng(12)
    w, h = 70, 67
    cs = _encode(rng.integers(0, 256, (h, w, 3), dtype=np.uint8), levels=2)
    want = S.J2kDecoder(cs, session).decode_to_numpy(S.PixelFormat.RGB8)
    pitch = 3 * w + pitch_extra
    base = S.DeviceSurface(session, pitch * h + 16, 1, S.PixelFormat.GRAY8)
    base.fill(0xC3)

    class Window:
        device_ptr, pitch_bytes, byte_len = base.device_ptr + offset, pitch, pitch * h

    plan = S.TilePlan(session, [cs], S.PixelFormat.RGB8, surfaces=[Window])
    assert _finals(plan) == ["9/7-rgb8"]
    plan.decode(S.MODE_GRAPH)
    session.synchronize()
    raw = base.to_numpy().reshape(-1)
    rows = raw[offset:offset + pitch * h].reshape(h, pitch)
    assert np.array_equal(rows[:, :3 * w].reshape(h, w, 3), want)
    assert (rows[:, 3 * w:] == 0xC3).all() and (raw[:offset] == 0xC3).all()
    assert (raw[offset + pitch * h:] == 0xC3).all()
    plan.close()
