"""The range that the 16-bit final stage of 8-bit RGB tiles rests on: streams whose
lower bands are scaled up (larger exponents in QCD) and come from two images, so
that the low-pass samples of the last level leave [-2048, 2048) in some 64x64 blocks
only, and bands of 11 and 12 bit-planes, against the oracle."""
import numpy as np
import pytest

import signinum_amd as S
from tests import oracle_ref as O

pytestmark = pytest.mark.gpu


def _lift(x, axis):
    """Forward 5/3 along an axis of even length and even origin: low, high."""
    x = np.moveaxis(x, axis, 0)
    e, o = x[0::2], x[1::2]
    d = o - ((e + np.concatenate([e[1:], e[-1:]])) >> 1)
    s = e + ((np.concatenate([d[:1], d[:-1]]) + d + 2) >> 2)
    return np.moveaxis(s, 0, axis), np.moveaxis(d, 0, axis)


def _unlift(s, d, axis):
    s, d = np.moveaxis(s, axis, 0), np.moveaxis(d, axis, 0)
    e = s - ((np.concatenate([d[:1], d[:-1]]) + d + 2) >> 2)
    o = d + ((e + np.concatenate([e[1:], e[-1:]])) >> 1)
    return np.moveaxis(np.stack([e, o], 1).reshape((-1,) + e.shape[1:]), 0, axis)


def _bands(luma):
    """LL, HL, LH and HH of the second level."""
    v_lo, v_hi = _lift(_lift(_lift(luma, 0)[0], 1)[0], 0)
    return [*_lift(v_lo, 1), *_lift(v_hi, 1)]


def _low_pass(a, b, shifts):
    """The last level's low-pass luma of a two-level decode with LL of a and the other
    lower bands of b, each of `shifts` more bit-planes."""
    luma = [v[..., 0].astype(np.int64) - 128 for v in (a, b)]
    bands = _bands(luma[0])[:1] + _bands(luma[1])[1:]
    for k, n in enumerate(shifts):
        if n:
            bands[k] = np.sign(bands[k]) * ((np.abs(bands[k]) << n) + (1 << (n - 1)))
    return _unlift(_unlift(bands[0], bands[1], 1), _unlift(bands[2], bands[3], 1), 0)


def _scaled(cs, shifts):
    """The codestream with larger exponents of the lowest bands."""
    cs = bytearray(cs)
    at = cs.index(b"\xff\x5c") + 5  # Lqcd 2, Sqcd 1
    assert cs[at - 1] & 0x1F == 0  # reversible: an exponent a band, in the top five bits
    for k, n in enumerate(shifts):
        cs[at + k] += n << 3
    return bytes(cs)


def _encode(img):
    return S.encode_j2k_ht(img, levels=2, use_mct=1, guard_bits=1, sop=1)


def _spliced(a, b):
    """a with the packets of the second resolution of b (one tile, LRCP, three
    components, an SOP marker before each packet)."""
    def packets(cs):
        sod = cs.index(b"\xff\x93") + 2
        at = [sod]
        for k in range(1, 9):
            at.append(cs.index(b"\xff\x91\x00\x04" + k.to_bytes(2, "big"), at[-1]))
        assert cs[at[0]:at[0] + 6] == b"\xff\x91\x00\x04\x00\x00"
        return cs[:sod], [cs[x:y] for x, y in zip(at, at[1:] + [len(cs) - 2])]
    head, pa = packets(a)
    pb = packets(b)[1]
    body = b"".join(pa[:3] + pb[3:6] + pa[6:])
    sot = head.index(b"\xff\x90")
    psot = len(head) - sot + len(body)
    return head[:sot + 6] + psot.to_bytes(4, "big") + head[sot + 10:] + body + a[-2:]


def _tile(seed, w, h):
    """Smooth gray, and saturated noise of 2x2 pixels in the middle.  (Gray: with one
    guard bit colours would not fit their bit-planes.)"""
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:h, 0:w]
    img = (128 + 40 * np.sin(x / 50 + seed) + 20 * np.cos(y / 37)).astype(np.uint8)
    n = rng.integers(0, 2, (64, 48)).astype(np.uint8) * 255
    y, x = (h - 128) // 4 * 2, (w - 96) // 4 * 2
    img[y:y + 128, x:x + 96] = n.repeat(2, 0).repeat(2, 1)
    return img[..., None].repeat(3, 2)


@pytest.mark.parametrize("w,h", [(512, 384), (260, 452)])
def test_low_pass_out_of_range_in_some_blocks(session, oracle, w, h):
    shifts = (3, 2, 2, 1)  # from 8, 9, 9 and 10 bit-planes to 11
    tiles = [_tile(k, w, h) for k in range(4)]
    coded = [_encode(v) for v in tiles]
    streams, past = [], 0
    for k in range(3):
        streams.append(_scaled(_spliced(coded[k], coded[k + 1]), shifts))
        # some 64x64 blocks have a low-pass sample past the range, most have none
        over = np.abs(_low_pass(tiles[k], tiles[k + 1], shifts)) > 2048
        blocks = [over[y:y + 32, x:x + 32].any() for y in range(0, h // 2, 32)
                  for x in range(0, w // 2, 32)]
        assert sum(blocks) < len(blocks) / 2
        past += sum(blocks)
    assert past >= 5
    plan = S.TilePlan(session, streams + coded[:1], S.PixelFormat.RGB8)
    assert [k for stage, k, _n in plan.kernels() if stage == "final"] == ["5/3-rgb8"]
    want = [O.decode(cs, 1) for cs in streams] + tiles[:1]
    for mode in (S.MODE_GRAPH, S.MODE_GRAPH, S.MODE_PLAIN):
        for s in plan.surfaces:
            s.fill(0x5A)
        plan.decode(mode)
        session.synchronize()
        for k, (s, ref) in enumerate(zip(plan.surfaces, want)):
            assert np.array_equal(s.to_numpy(), ref), (mode, k)
    plan.close()


@pytest.mark.parametrize("planes,kernel", [(11, "5/3-rgb8"), (12, "5/3-general")])
def test_bit_planes_of_either_kernel(session, oracle, planes, kernel):
    """Noise in every band, HH with 11 and with 12 bit-planes."""
    img = np.random.default_rng(planes).integers(0, 2, (200, 150, 3), dtype=np.uint8) * 255
    cs = S.encode_j2k_ht(img, levels=2, use_mct=1)
    at = cs.index(b"\xff\x5c") + 5
    assert max(cs[at:at + 7]) >> 3 == 10 and cs[at - 1] >> 5 == 2  # HH: 10 + 2 - 1 = 11
    cs = _scaled(cs, (0, 0, 0, planes - 11, 0, 0, planes - 11))
    plan = S.TilePlan(session, [cs], S.PixelFormat.RGB8)
    assert [k for stage, k, _n in plan.kernels() if stage == "final"] == [kernel]
    plan.decode(S.MODE_GRAPH)
    session.synchronize()
    assert np.array_equal(plan.surfaces[0].to_numpy(), O.decode(cs, 1))
    plan.close()
