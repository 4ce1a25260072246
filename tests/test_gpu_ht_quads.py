"""The split HT kernels with four lanes a block (lists of blocks at most 16 wide)
where their pairs, groups, rings and work-groups end: every width up to 16,
heights up to 64, lists that fill neither a wave nor a work-group, int16 and int32
samples, refinement passes with and without stripe-causal contexts, damaged
bytes, against the source or the oracle."""
import numpy as np
import pytest

import signinum_amd as S
from tests import oracle_ref as O
from tests.test_gpu_ht_refine_split import _causal, _content

pytestmark = pytest.mark.gpu


def _check(session, streams, want, fmt, quads=True):
    plan = S.TilePlan(session, streams, fmt)
    for v, name in enumerate(S.TilePlan.lane_variants()):
        plan.lane_variant = v
        kernel = [k for stage, k, _n in plan.kernels() if stage == "blocks"]
        assert kernel == [name + ("-quads" if quads and name != "wave-coop" else "")]
        for s in plan.surfaces:
            s.fill(0xA5)
        plan.decode(S.MODE_GRAPH)
        session.synchronize()
        for k, (s, ref) in enumerate(zip(plan.surfaces, want)):
            assert np.array_equal(s.to_numpy(), ref), (name, k)
    plan.close()


@pytest.mark.parametrize("depth", [8, 16])
@pytest.mark.parametrize("kind", ["noise", "sparse"])
@pytest.mark.parametrize("refine", [0, 1, 2])
def test_narrow_blocks(session, oracle, kind, depth, refine):
    rng = np.random.default_rng(depth + refine)
    streams, want = [], []
    fmt = S.PixelFormat.GRAY8 if depth == 8 else S.PixelFormat.GRAY16
    for w, h, cbw, cbh, levels in [(1, 1, 2, 2, 0), (2, 3, 4, 6, 0), (4, 4, 2, 2, 0), (5, 64, 4, 6, 0),
                                   (11, 9, 3, 4, 0), (12, 63, 4, 6, 0), (13, 62, 4, 6, 0),
                                   (15, 64, 4, 6, 0), (16, 64, 4, 6, 0), (17, 65, 4, 6, 0),
                                   (61, 130, 4, 6, 2), (100, 37, 2, 4, 1), (77, 90, 4, 2, 3)]:
        img = _content(kind, rng, w, h, depth)
        cs = S.encode_j2k_ht(img, bit_depth=depth, levels=levels, cb_width_log2=cbw,
                             cb_height_log2=cbh, use_mct=0, ht_refine=refine)
        for c in (cs, _causal(cs)) if refine else (cs,):
            streams.append(c)
            want.append(O.decode(c, int(fmt)) if refine else img[..., None])
    _check(session, streams, want, fmt)
    _check(session, streams[2:3] * 7, want[2:3] * 7, fmt)


def test_lists_with_a_wider_block(session, oracle):
    rng = np.random.default_rng(2)
    imgs = [rng.integers(0, 256, (40, w), dtype=np.uint8) for w in (16, 17)]
    streams = [S.encode_j2k_ht(v, levels=0, cb_width_log2=5, use_mct=0) for v in imgs]
    _check(session, streams, [v[..., None] for v in imgs], S.PixelFormat.GRAY8, quads=False)


@pytest.mark.parametrize("refine", [0, 2])
def test_damaged_blocks_decode_as_the_oracle_does(session, oracle, refine):
    rng = np.random.default_rng(8 + refine)
    cs = S.encode_j2k_ht(_content("noise", rng, 96, 80, 8), levels=1, use_mct=0, ht_refine=refine,
                         cb_width_log2=4, cb_height_log2=6)
    start, good, failed = cs.index(b"\xff\x93") + 100, [], 0
    for k in range(60):
        bad = bytearray(cs)
        at, n = int(rng.integers(start, len(cs) - 40)), int(rng.integers(1, 24))
        bad[at:at + n] = (b"\xff" * n if k % 2 else
                          rng.choice([0x7F, 0xFF, 0x90, 0x00], n).astype(np.uint8).tobytes())
        if O.decode_rc(bytes(bad), int(S.PixelFormat.GRAY8)) == 0:
            good.append(bytes(bad))
        else:
            failed += 1
            with pytest.raises((S.J2kError, S.TileBatchError)):
                S.decode_tiles_to_device(session, [bytes(bad)], S.PixelFormat.GRAY8)
    assert good
    _check(session, good, [O.decode(c, int(S.PixelFormat.GRAY8)) for c in good],
           S.PixelFormat.GRAY8)
