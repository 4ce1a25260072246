"""Which classic kernel a list takes (block shape and blocks per CU), and that
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


@pytest.mark.parametrize("exps,per_cu,kernel", [
    ((6, 6), 1, "usual-l1"), ((6, 6), 45, "usual-l1"), ((6, 6), 48, "usual-l3"),
    ((6, 6), 270, "usual-l3"), ((6, 6), 290, "rows-w64"),
    ((5, 5), 20, "small-l1"), ((5, 5), 40, "small-l2"), ((5, 5), 100, "small-l4"),
    ((5, 5), 300, "small-l16"), ((5, 5), 470, "rows-w32"),
    ((7, 5), 1, "long-l1"), ((7, 5), 40, "long-l1"), ((7, 5), 50, "rows-w256")])
def test_kernel_of_a_list(session, exps, per_cu, kernel):
    plan, imgs = _plan(session, *exps, blocks=per_cu * CUS)
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
    ("64", "rows-w64", "rows-w32", "rows-w256"), ("32", "rows-w64", "rows-w32", "rows-w256"),
    ("16", "rows-w64", "small-l16", "rows-w256"), ("4", "usual-l1", "small-l4", "long-l1"),
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
