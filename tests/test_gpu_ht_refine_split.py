"""The refinement kernels (prepare, SigProp chain, apply) where their tiles
end: sides around the groups, stripes and lanes of a block, lists that fill
neither a wave nor a work-group, stripe-causal contexts, int16 and int32
samples, and passes over damaged bytes (0xFF runs: stuffing in every place),
against the oracle."""
import numpy as np
import pytest

import signinum_amd as S
from tests import oracle_ref as O

pytestmark = pytest.mark.gpu


def _content(kind, rng, w, h, depth):
    top = 1 << depth
    dt = np.uint8 if depth == 8 else np.uint16
    if kind == "noise":
        return rng.integers(0, top, (h, w)).astype(dt)
    img = np.full((h, w), top // 2, dt)  # sparse: few members, found one after another
    n = max(1, w * h // 30)
    img[rng.integers(0, h, n), rng.integers(0, w, n)] = rng.integers(0, top, n)
    return img


def _causal(cs):
    """The codestream with the stripe-causal bit of its code-block style set."""
    cs = bytearray(cs)
    at = cs.index(b"\xff\x52") + 12  # COD: Lcod 2, Scod 1, SGcod 4, levels, xcb, ycb
    assert cs[at] & 0x40
    cs[at] |= 0x08
    return bytes(cs)


def _check(session, streams, fmt):
    plan = S.TilePlan(session, streams, fmt)
    want = [O.decode(cs, int(fmt)) for cs in streams]
    for v, name in enumerate(S.TilePlan.lane_variants()):
        plan.lane_variant = v
        for s in plan.surfaces:
            s.fill(0xA5)
        plan.decode(S.MODE_GRAPH)
        session.synchronize()
        for k, (s, ref) in enumerate(zip(plan.surfaces, want)):
            assert np.array_equal(s.to_numpy(), ref), (name, k)
    plan.close()


@pytest.mark.parametrize("depth", [8, 16])
@pytest.mark.parametrize("kind", ["noise", "sparse"])
@pytest.mark.parametrize("refine", [1, 2])
def test_block_edges(session, oracle, kind, refine, depth):
    rng = np.random.default_rng(31 * depth + refine)
    streams = []
    for w, h, cbw, cbh, levels in [(1, 1, 2, 2, 0), (3, 5, 2, 2, 0), (4, 4, 2, 2, 0), (5, 9, 3, 4, 0),
                                   (33, 31, 6, 6, 0), (60, 62, 6, 6, 0), (61, 63, 6, 6, 0),
                                   (64, 64, 6, 6, 0), (65, 66, 6, 6, 0), (127, 130, 5, 6, 2),
                                   (200, 8, 6, 2, 1), (9, 210, 3, 6, 1)]:
        cs = S.encode_j2k_ht(_content(kind, rng, w, h, depth), bit_depth=depth, levels=levels,
                             cb_width_log2=cbw, cb_height_log2=cbh, use_mct=0, ht_refine=refine)
        streams += [cs, _causal(cs)]
    _check(session, streams, S.PixelFormat.GRAY8 if depth == 8 else S.PixelFormat.GRAY16)


def test_damaged_passes_decode_as_the_oracle_does(session, oracle):
    rng = np.random.default_rng(8)
    cs = S.encode_j2k_ht(_content("noise", rng, 128, 120, 8), levels=1, use_mct=0, ht_refine=2)
    start, good = cs.index(b"\xff\x93") + 100, []
    for k in range(60):
        bad = bytearray(cs)
        at, n = int(rng.integers(start, len(cs) - 40)), int(rng.integers(1, 24))
        bad[at:at + n] = (b"\xff" * n if k % 2 else
                          rng.choice([0x7F, 0xFF, 0x90, 0x00], n).astype(np.uint8).tobytes())
        if O.decode_rc(bytes(bad), int(S.PixelFormat.GRAY8)) == 0:
            good.append(bytes(bad))
    assert good
    _check(session, good, S.PixelFormat.GRAY8)
