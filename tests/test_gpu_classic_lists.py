"""Which classic kernel a list takes (block shape, costs and blocks per CU), and that
each one decodes full-size blocks: 64x64, 32x32, and the long shapes (more than
128 groups of 8x4 samples) with and without raw segments, against the source."""
import numpy as np
import pytest

import signinum_amd as S

pytestmark = pytest.mark.gpu

CUS = 256  # compute units of an MI355X


def _plan(session, cbw, cbh, blocks, style=0, side=512):
    """At least `blocks` code-blocks of 2^cbw x 2^cbh samples, nothing else."""
    rng = np.random.default_rng(cbw + style)
    w, h = max(side, 1 << cbw), max(side, 1 << cbh)
    imgs = [rng.integers(0, 256, (h, w, 1), dtype=np.uint8),
            (rng.integers(0, 4, (h, w, 1)) + np.arange(w)[:, None] // 8 % 64).astype(np.uint8)]
    streams = [S.encode_j2k_classic(v, cb_style=style, cb_width_log2=cbw, cb_height_log2=cbh,
                                    levels=0, use_mct=0) for v in imgs]
    n = -(-blocks // ((w >> cbw) * (h >> cbh)))
    return S.TilePlan(session, [streams[k % 2] for k in range(n)], S.PixelFormat.GRAY8), imgs


def _kernels(plan):
    return [k for stage, k, _n in plan.kernels() if stage == "classic"]


def _check(session, plan, imgs):
    n = len(plan.surfaces)
    for s in plan.surfaces:
        s.fill(0x5A)
    plan.decode(S.MODE_GRAPH)
    session.synchronize()
    for k in sorted({0, 1, n // 2, n - 1} & set(range(n))):
        assert np.array_equal(plan.surfaces[k].to_numpy(), imgs[k % 2]), k


@pytest.mark.parametrize("exps,style,per_cu,kernel", [
    ((6, 6), 0, 1, "usual-l1"), ((6, 6), 0, 16, "usual-l3"), ((6, 6), 0, 130, "rows-w64-l32"),
    ((5, 5), 0, 1, "small-l1"), ((5, 5), 0, 15, "small-l2"), ((5, 5), 0, 30, "small-l4"),
    ((5, 5), 0, 90, "small-l16"), ((5, 5), 0, 150, "rows-w32-l32"), ((5, 5), 0, 600, "rows-w32-l64"),
    ((7, 5), 0, 1, "long-l1"), ((7, 5), 0, 80, "rows-w256-l32"),
    ((6, 6), 1, 1, "usual-raw-l1"), ((6, 6), 1, 16, "usual-raw-l3"), ((6, 6), 1, 130, "rows-w64-l32"),
    ((5, 5), 1, 1, "small-raw-l1"), ((5, 5), 1, 16, "small-raw-l2"), ((5, 5), 1, 30, "small-raw-l4"),
    ((5, 5), 1, 90, "small-raw-l16"), ((5, 5), 1, 600, "rows-w32-l64"), ((7, 5), 1, 1, "long-raw-l1")])
def test_kernel_of_a_list(session, exps, style, per_cu, kernel):
    plan, imgs = _plan(session, *exps, blocks=per_cu * CUS, style=style)
    assert _kernels(plan) == [kernel]
    _check(session, plan, imgs)
    plan.close()


@pytest.mark.parametrize("exps,style,kernel", [
    ((7, 5), 0, "long-l1"), ((8, 4), 0, "long-l1"), ((9, 3), 0, "long-l1"), ((10, 2), 0, "long-l1"),
    ((2, 10), 0, "long-l1"), ((5, 7), 0, "usual-l1"), ((7, 5), 1, "long-raw-l1"),
    ((10, 2), 1, "long-raw-l1"), ((2, 10), 1 | 4, "long-raw-l1"), ((7, 5), 2 | 8 | 0x20, "long-l1")])
def test_long_blocks(session, exps, style, kernel):
    plan, imgs = _plan(session, *exps, blocks=40, style=style, side=256)
    assert _kernels(plan) == [kernel]
    _check(session, plan, imgs)
    plan.close()


@pytest.mark.parametrize("lanes,usual,small,long", [
    ("64", "rows-w64-l32", "rows-w32-l64", "rows-w256-l32"),
    ("32", "rows-w64-l32", "rows-w32-l64", "rows-w256-l32"),
    ("16", "rows-w64-l32", "small-l16", "rows-w256-l32"),
    ("r32", "rows-w64-l32", "rows-w32-l32", "rows-w256-l32"),
    ("r16", "usual-l1", "rows-w32-l16", "long-l1"), ("4", "usual-l1", "small-l4", "long-l1"),
    ("3", "usual-l3", "small-l1", "long-l1"), ("1", "usual-l1", "small-l1", "long-l1"),
    ("5", "usual-l1", "small-l1", "long-l1")])
def test_forced_lanes(session, monkeypatch, lanes, usual, small, long):
    """A forced count names a kernel of the shape, or the row kernels, or nothing."""
    monkeypatch.setenv("SGN_CLASSIC_LANES", lanes)
    for exps, kernel in (((6, 6), usual), ((5, 5), small), ((7, 5), long)):
        plan, imgs = _plan(session, *exps, blocks=70, side=256)
        assert _kernels(plan) == [kernel]
        _check(session, plan, imgs)
        plan.close()


@pytest.mark.parametrize("style", [0, 1])
def test_widest_rows(session, monkeypatch, style):
    """The row kernel of blocks over 256 wide, at full size."""
    monkeypatch.setenv("SGN_CLASSIC_LANES", "32")
    plan, imgs = _plan(session, 10, 2, blocks=40, style=style, side=64)
    assert _kernels(plan) == ["rows-w1024-l16"]
    _check(session, plan, imgs)
    plan.close()
