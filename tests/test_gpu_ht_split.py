"""The split HT cleanup (clean, symbols, magnitudes) where its tiles end:
block sides around the pair, segment and row limits of its lanes, lists that
fill neither a wave nor a work-group, streams rich in 0xFF and in long MEL
runs, int32 samples, and damaged code-block data, against the oracle."""
import numpy as np
import pytest

import signinum_amd as S
from signinum_amd import synth
from tests import oracle_ref as O

pytestmark = pytest.mark.gpu

SPLIT = [n for n in ("split-l64", "split-l32")]


def _decode(session, streams, fmt, variant, mode=S.MODE_GRAPH):
    plan = S.TilePlan(session, streams, fmt)
    plan.lane_variant = S.TilePlan.lane_variants().index(variant)
    for s in plan.surfaces:
        s.fill(0xA5)
    plan.decode(mode)
    session.synchronize()
    out = [s.to_numpy() for s in plan.surfaces]
    plan.close()
    return out


def _content(kind, rng, w, h):
    if kind == "noise":  # full-range noise: MagSgn bytes of 0xFF
        return rng.integers(0, 256, (h, w), dtype=np.uint8)
    if kind == "sparse":  # few significant quads: MEL runs of every length
        img = np.full((h, w), 128, np.uint8)
        n = max(1, w * h // 50)
        img[rng.integers(0, h, n), rng.integers(0, w, n)] = rng.integers(0, 256, n)
        return img
    return np.full((h, w), 77, np.uint8)  # flat: blocks without coded data


@pytest.mark.parametrize("variant", SPLIT)
@pytest.mark.parametrize("kind", ["noise", "sparse", "flat"])
@pytest.mark.parametrize("w,h,cbw,cbh,levels", [
    (1, 1, 2, 2, 0), (3, 5, 2, 2, 0), (4, 4, 2, 2, 0),      # one pair, one lane
    (29, 31, 5, 5, 0), (32, 33, 5, 5, 1), (33, 64, 6, 6, 0),  # around one segment of a row
    (35, 63, 6, 6, 0), (61, 7, 6, 4, 0), (62, 62, 6, 6, 0),
    (63, 64, 6, 6, 0), (64, 64, 6, 6, 0), (65, 66, 6, 6, 0),  # a full block and what hangs over
    (127, 129, 6, 6, 3), (200, 8, 6, 2, 1), (9, 210, 3, 6, 1),
])
def test_block_edges(session, oracle, variant, kind, w, h, cbw, cbh, levels):
    img = _content(kind, np.random.default_rng(w * 1000 + h), w, h)
    cs = S.encode_j2k_ht(img, levels=levels, cb_width_log2=cbw, cb_height_log2=cbh, use_mct=0)
    got = _decode(session, [cs], S.PixelFormat.GRAY8, variant)[0]
    assert np.array_equal(got[..., 0], img)


@pytest.mark.parametrize("variant", SPLIT)
def test_int32_samples_and_lists_of_every_remainder(session, oracle, variant):
    """16-bit samples of full range (31 bits a sample at most), 1 to 9 tiles
    of 35 blocks each: the last group, wave and work-group partly filled."""
    rng = np.random.default_rng(5)
    imgs = [rng.integers(0, 65536, (150, 70 + k), dtype=np.uint16) for k in range(9)]
    streams = [S.encode_j2k_ht(v, bit_depth=16, use_mct=0, levels=2, cb_width_log2=5,
                               cb_height_log2=4) for v in imgs]
    for n in (1, 2, 3, 9):
        for got, want in zip(_decode(session, streams[:n], S.PixelFormat.GRAY16, variant), imgs):
            assert np.array_equal(got[..., 0], want)


def test_order_that_needs_more_workspace(session, oracle):
    """Reordering a plan lays its workspace out again (a group of 64 blocks
    reserves its largest block's size for each): every order decodes."""
    streams, pix, _cls = synth.lossless_batch_with_pixels(20, size=200)
    plan = S.TilePlan(session, streams, S.PixelFormat.RGB8)
    for order in (1, 0, 4, 3, 1):
        plan.order_code_blocks(order)
        for s in plan.surfaces:
            s.fill(0)
        plan.decode(S.MODE_GRAPH)
        session.synchronize()
        assert all(np.array_equal(s.to_numpy(), v) for s, v in zip(plan.surfaces, pix)), order
    plan.close()


@pytest.mark.parametrize("variant", SPLIT + ["wave-coop"])
def test_damaged_blocks_decode_as_the_oracle_does(session, oracle, variant):
    """Bytes of the code-block data overwritten (0xFF runs, random values):
    where the oracle decodes, so does the device, to the same pixels; where it
    reports a failing block, so does the device."""
    rng = np.random.default_rng(99)
    img = synth.texture_rgb(rng, 150, 130)
    cs = S.encode_j2k_lossless(img, levels=2)
    start = cs.index(b"\xff\x93") + 400
    same = failed = 0
    for k in range(24):
        bad = bytearray(cs)
        for _ in range(1 + k % 4):
            at = int(rng.integers(start, len(bad) - 40))
            n = int(rng.integers(1, 16))
            bad[at:at + n] = b"\xff" * n if k % 3 == 0 else rng.integers(0, 255, n, dtype=np.uint8).tobytes()
        bad = bytes(bad)
        if O.decode_rc(bad, 1) == 0:
            got = _decode(session, [bad], S.PixelFormat.RGB8, variant)[0]
            assert np.array_equal(got, O.decode(bad, 1)), k
            same += 1
        else:
            failed += 1
            with pytest.raises((S.J2kError, S.TileBatchError)):
                S.decode_tiles_to_device(session, [bad], S.PixelFormat.RGB8)
    assert same


def test_former_variant_indexes(session):
    """Indexes 0 to 8 are accepted and decode; 9 and -1 are refused."""
    img = np.random.default_rng(4).integers(0, 256, (70, 90, 3), dtype=np.uint8)
    plan = S.TilePlan(session, [S.encode_j2k_lossless(img)], S.PixelFormat.RGB8)
    names, own = S.TilePlan.lane_variants(), plan.lane_variant
    for v in range(9):
        plan.lane_variant = v
        want = v if v < len(names) else names.index("wave-coop") if v == 6 else own
        assert plan.lane_variant == want
        plan.surfaces[0].fill(0x5A)
        plan.decode(S.MODE_GRAPH)
        session.synchronize()
        assert np.array_equal(plan.surfaces[0].to_numpy(), img), v
    for v in (-1, 9):
        with pytest.raises(S.J2kError):
            plan.lane_variant = v
    plan.close()
