"""Decodes into host arrays: the pinned download where its chunks (8 MB, whole
rows) and pieces (256 KB) end, strided arrays, arrays that cannot take their
tile, failing tiles, and calls in turn on one session (its device blocks and
pinned memory are reused)."""
import numpy as np
import pytest

import signinum_amd as S
from signinum_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tiles():
    rng = np.random.default_rng(31)
    imgs = [synth.texture_rgb(rng, w, h) for w, h in ((256, 256), (1, 1), (301, 77), (64, 300))]
    return imgs, [S.encode_j2k_lossless(v, levels=2) for v in imgs]


@pytest.mark.parametrize("pad", [0, 1, 13])
def test_strided_tiles_and_regions(session, tiles, pad):
    imgs, streams = tiles
    outs = [np.full(v.shape[0] * (v.shape[1] * 3 + pad), 0xEE, np.uint8) for v in imgs]
    S.decode_tiles_into([(c, o, v.shape[1] * 3 + pad) for c, o, v in zip(streams, outs, imgs)],
                        S.PixelFormat.RGB8, session=session)
    for o, v in zip(outs, imgs):
        rows = o.reshape(v.shape[0], -1)
        assert np.array_equal(rows[:, :v.shape[1] * 3].reshape(v.shape), v)
        assert (rows[:, v.shape[1] * 3:] == 0xEE).all()
    v = imgs[2]
    roi = (17, 5, 200, 60)
    out = np.full(60 * (600 + pad), 0xEE, np.uint8)
    S.decode_tiles_region_scaled_into([(streams[2], out, 600 + pad, roi, S.Downscale.NONE)],
                                      S.PixelFormat.RGB8, session=session)
    rows = out.reshape(60, -1)
    assert np.array_equal(rows[:, :600].reshape(60, 200, 3), v[5:65, 17:217])
    assert (rows[:, 600:] == 0xEE).all()


def test_more_than_two_chunks_and_batches_in_turn(session, tiles):
    """150 tiles of 196 KB (30 MB: four chunks), then a call of another size,
    then the first again, on one session; pipelined in chunks of tiles too."""
    imgs, streams = tiles
    for n in (150, 3, 150):
        outs = [np.zeros(imgs[0].size, np.uint8) for _ in range(n)]
        S.decode_tiles_into([(streams[0], o, 768) for o in outs], S.PixelFormat.RGB8, session=session)
        assert all(np.array_equal(o.reshape(imgs[0].shape), imgs[0]) for o in outs)
    big = synth.near_white_rgb(np.random.default_rng(2), 2500, 1300)  # one image over a chunk
    out = S.J2kDecoder(S.encode_j2k_lossless(big), session).decode_to_numpy(S.PixelFormat.RGB8)
    assert np.array_equal(out, big)


def test_pipelined_into_host(session, tiles, monkeypatch):
    monkeypatch.setenv("SGN_PIPELINE_TILES", "5")
    imgs, streams = tiles
    outs = [np.zeros(imgs[k % 4].size, np.uint8) for k in range(23)]
    S.decode_tiles_into([(streams[k % 4], o, imgs[k % 4].shape[1] * 3) for k, o in enumerate(outs)],
                        S.PixelFormat.RGB8, session=session)
    assert all(np.array_equal(o.reshape(imgs[k % 4].shape), imgs[k % 4]) for k, o in enumerate(outs))


def test_small_array_and_failing_tile(session, tiles):
    imgs, streams = tiles
    outs = [np.zeros(v.size, np.uint8) for v in imgs]
    small = np.zeros(imgs[2].size - 1, np.uint8)
    with pytest.raises(S.J2kError):
        S.decode_tiles_into([(streams[0], outs[0], 768), (streams[2], small, 903)],
                            S.PixelFormat.RGB8, session=session)
    assert np.array_equal(outs[0].reshape(imgs[0].shape), imgs[0])  # the tile before it is written
    outs[0][:] = 7
    for bad in (streams[2][:60], b"\xff\x4f\xff\x51 no image"):
        with pytest.raises(S.TileBatchError) as e:
            S.decode_tiles_into([(streams[0], outs[0], 768), (bad, outs[2], 903)],
                                S.PixelFormat.RGB8, session=session)
        assert e.value.index == 1 and (outs[0] == 7).all()
    with pytest.raises(S.J2kError):
        ro = np.zeros(imgs[0].size, np.uint8)
        ro.flags.writeable = False
        S.decode_tiles_into([(streams[0], ro, 768)], S.PixelFormat.RGB8, session=session)
    S.decode_tiles_into([], S.PixelFormat.RGB8, session=session)


def test_arrays_that_share_bytes_and_one_canvas(session):
    """Tiles decoded into one array: the last one stays.  Tiles of one canvas
    (flat views that overlap in range only) land in their places."""
    rng = np.random.default_rng(9)
    imgs = [synth.texture_rgb(rng, 256, 256) for _ in range(64)]
    streams = [S.encode_j2k_lossless(v, levels=2) for v in imgs]
    for _ in range(3):
        out = np.zeros(imgs[0].size, np.uint8)
        S.decode_tiles_into([(c, out, 768) for c in streams], S.PixelFormat.RGB8, session=session)
        assert np.array_equal(out.reshape(256, 256, 3), imgs[-1])
    canvas = np.zeros((8 * 256, 8 * 256, 3), np.uint8)
    flat = canvas.reshape(-1)
    pitch = 8 * 768
    S.decode_tiles_into([(c, flat[(k // 8) * 256 * pitch + (k % 8) * 768:], pitch)
                         for k, c in enumerate(streams)], S.PixelFormat.RGB8, session=session)
    for k, v in enumerate(imgs):
        y, x = 256 * (k // 8), 256 * (k % 8)
        assert np.array_equal(canvas[y:y + 256, x:x + 256], v), k


@pytest.mark.parametrize("pad", [0, 13])
def test_page_locked_arrays(session, tiles, pad):
    """Downloads and decodes into page-locked memory, tight and strided."""
    import ctypes

    from signinum_amd import _lib
    imgs, streams = tiles
    L = _lib.load()
    p = ctypes.c_void_p()
    size = max((v.shape[1] * 3 + pad) * v.shape[0] for v in imgs)
    assert L.sgn_host_alloc(size, ctypes.byref(p)) == 0
    try:
        mem = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_uint8)), (size,))
        for v, c in zip(imgs, streams):
            stride = v.shape[1] * 3 + pad
            out = mem[:stride * v.shape[0]]
            surf = S.J2kDecoder(c, session).submit_to_device(session, S.PixelFormat.RGB8)
            for write in (lambda: surf.download_into(out, stride),
                          lambda: S.decode_tiles_into([(c, out, stride)], S.PixelFormat.RGB8,
                                                      session=session)):
                out[:] = 0xEE
                write()
                rows = out.reshape(v.shape[0], stride)
                assert np.array_equal(rows[:, :v.shape[1] * 3].reshape(v.shape), v)
                assert (rows[:, v.shape[1] * 3:] == 0xEE).all()
    finally:
        L.sgn_host_free(p)
