"""Decode workloads that are timed: what a program that reads JPEG 2000 tiles
does with this package, over the sizes, coders and sample types it meets.

Three entry points are called:

* `replay`: a `TilePlan` whose codestreams are resident in device memory,
  decoded as a graph into surfaces the program owns (a torch tensor).  This
  is the loop of bench.py and of a viewer or a training loader that keeps its
  coded tiles on the GPU.
* `tiles`: `decode_tiles_into`, host codestreams to host arrays, one batch.
* `tile` / `region`: `J2kDecoder.decode_to_numpy` and
  `decode_region_to_numpy`, one codestream to one host array.

Every case is a dict of plain values; `prepare` draws pixels from the seed,
encodes them with the package's encoder and builds what the program keeps.
Geometry depends on the case alone, pixels on the seed alone.  A batch cycles
through a pool of distinct tiles; each of its tiles has its own copy of the
coded bytes and its own output.
"""
import random
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import signinum_amd as S
from signinum_amd import synth

_BASE = {
    "call": "replay",
    "coder": "ht",       # ht, ht-refined (SigProp + MagRef in every block), classic
    "wavelet": "5/3",    # 5/3 (lossless, RCT) or 9/7 (lossy, ICT)
    "content": "slide",  # slide, tissue, spots12, gray16, mixed
    "tiles": 1, "pool": 1, "width": 256, "height": 256,
    "levels": 5, "block": 6, "scale": 1, "tile_side": 0,
    "roi_x": 0, "roi_y": 0, "roi_w": 0, "roi_h": 0,
}


def _case(**kw):
    return {**_BASE, **kw}


def listed():
    return [
        # One tile read on its own, file bytes to pixels: a slide viewer's
        # first paint, and the smallest call a program makes.
        _case(name="tile-256", call="tile"),
        # A viewport cut out of a slide level that is not a multiple of
        # anything, at half resolution.
        _case(name="region-half", call="region", width=1700, height=1200, content="tissue", pool=1,
              scale=2, roi_x=233, roi_y=151, roi_w=1201, roi_h=803),
        # A page of tiles, host bytes to host arrays.
        _case(name="tiles-host-240", call="tiles", tiles=240, pool=60, width=240, height=240),
        # One 512x512 tile already on the GPU: the latency of a decode.
        _case(name="one-512", content="tissue", width=512, height=512),
        # A viewer's screen: 24 tiles in one request.
        _case(name="screen-24", tiles=24, pool=24),
        # A training batch of ordinary size.
        _case(name="batch-384", tiles=384, pool=64),
        # The headline batch: a slide's worth of 256x256 tiles.
        _case(name="batch-4096", tiles=4096, pool=96),
        # Lossy slides: 9/7 + ICT in f32, 512x512 tiles.
        _case(name="lossy-192", wavelet="9/7", content="tissue", tiles=192, pool=32, width=512,
              height=512),
        # 16-bit gray frames of odd sizes (32-bit coefficients all the way).
        _case(name="gray16-12", content="gray16", tiles=12, pool=6, width=1001, height=777),
        # One plan of several geometries, bit depths, block sizes and scales.
        _case(name="mixed-160", content="mixed", tiles=160, pool=40),
        # HTJ2K with refinement passes in every code-block.
        _case(name="refined-512", coder="ht-refined", tiles=512, pool=48),
        # Part 1 (EBCOT / MQ) tiles: what existing archives hold.
        _case(name="classic-256", coder="classic", tiles=256, pool=32),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case of the same ranges: any call, coder and content, tile
    counts and sides spread over their logarithms, odd sizes among them."""
    kind = rng.choice(["tile", "region", "tiles", "replay", "replay", "replay", "lossy", "gray16",
                       "spots12", "mixed", "refined", "classic"])
    side = lambda lo, hi: _log(rng, lo, hi)  # noqa: E731
    block = rng.choice([5, 6, 6])
    levels = rng.randint(3, 6)
    if kind == "tile":
        return _case(call="tile", content=rng.choice(["slide", "tissue"]), width=side(100, 1200),
                     height=side(100, 1200), block=block, levels=levels, scale=rng.choice([1, 1, 2]))
    if kind == "region":
        w, h = side(600, 1900), side(600, 1500)
        rw, rh = side(64, w // 2), side(64, h // 2)
        return _case(call="region", content="tissue", width=w, height=h, block=block,
                     levels=levels, scale=rng.choice([1, 2, 4]), roi_x=rng.randrange(w - rw),
                     roi_y=rng.randrange(h - rh), roi_w=rw, roi_h=rh,
                     tile_side=rng.choice([0, 0, 512]))
    if kind == "tiles":
        n = _log(rng, 8, 1000)
        return _case(call="tiles", tiles=n, pool=min(n, 48), width=side(128, 300),
                     height=side(128, 300), block=block, levels=levels)
    if kind == "gray16":
        n = _log(rng, 1, 24)
        return _case(content="gray16", tiles=n, pool=min(n, 4), width=side(256, 1200),
                     height=side(256, 1200), block=block, levels=levels)
    if kind == "spots12":
        n = _log(rng, 1, 200)
        return _case(content="spots12", tiles=n, pool=min(n, 12), width=side(128, 512),
                     height=side(128, 512), block=block, levels=levels, scale=rng.choice([1, 2]))
    if kind == "lossy":
        n = _log(rng, 1, 200)
        return _case(wavelet="9/7", content="tissue", tiles=n, pool=min(n, 16), width=side(200, 640),
                     height=side(200, 640), block=block, levels=levels)
    if kind == "mixed":
        n = _log(rng, 16, 200)
        return _case(content="mixed", tiles=n, pool=min(n, 40))
    if kind == "refined":
        n = _log(rng, 4, 512)
        return _case(coder="ht-refined", tiles=n, pool=min(n, 32), width=side(128, 300),
                     height=side(128, 300), levels=levels)
    if kind == "classic":
        n = _log(rng, 1, 256)
        return _case(coder="classic", tiles=n, pool=min(n, 24), width=side(128, 256),
                     height=side(128, 256), block=block, levels=levels)
    n = _log(rng, 1, 2500)
    return _case(tiles=n, pool=min(n, 64), width=side(150, 300), height=side(150, 300), block=block,
                 levels=levels)


# ---- inputs -----------------------------------------------------------------

_SLIDE = (1, 0, 1, 2, 1, 0, 1, 2, 1, 0)  # 30% near-white, 50% tissue, 20% texture


def _geometry(case, i):
    """(width, height, levels, block exponent, scale, content) of pool tile i."""
    if case["content"] != "mixed":
        return (case["width"], case["height"], case["levels"], case["block"], case["scale"],
                case["content"])
    r = random.Random(1000 + i)
    size = (240, 256, 512, 1024)[i % 4]
    return (size, size, r.randint(3, 6), r.choice([5, 6]), r.choice([1, 2, 4]),
            r.choice(["slide", "slide", "slide", "spots12"]))


def _pixels(content, rng, i, w, h):
    if content == "spots12":
        return synth.spots_gray12(rng, w, h), 12
    if content == "gray16":
        # a radiograph: a smooth field over most of the 16-bit range, with noise
        y, x = np.mgrid[0:h, 0:w].astype(np.float64)
        a, b, c = rng.uniform(2, 6, 3)
        f = np.sin(a * x / w + b) * np.cos(c * y / h) * 20000 + 32768
        return np.clip(np.rint(f + rng.normal(0, 60, (h, w))), 0, 65535).astype(np.uint16), 16
    if content == "tissue":
        return synth.tissue_rgb(rng, w, h), 8
    make = (synth.near_white_rgb, synth.tissue_rgb, synth.texture_rgb)[_SLIDE[i % len(_SLIDE)]]
    return make(rng, w, h), 8


def _pool_tile(case, seed, i):
    w, h, levels, block, scale, content = _geometry(case, i)
    img, bits = _pixels(content, synth.tile_rng(seed, i), i, w, h)
    opts = dict(bit_depth=bits, levels=levels, cb_width_log2=block, cb_height_log2=block,
                use_mct=1 if img.ndim == 3 else 0)
    if case["tile_side"]:
        opts.update(tile_width=case["tile_side"], tile_height=case["tile_side"])
    if case["wavelet"] == "9/7":
        opts.update(reversible=0, base_step=1.0 / 64, guard_bits=2)
    if case["coder"] == "ht-refined":
        opts.update(ht_refine=2)
    encode = S.encode_j2k_classic if case["coder"] == "classic" else S.encode_j2k_ht
    fmt = S.PixelFormat.RGB8 if bits == 8 else S.PixelFormat.GRAY16
    return encode(img, **opts), fmt, S.Downscale(scale), img


def _pool(case, seed):
    with ThreadPoolExecutor(16) as ex:
        return list(ex.map(lambda i: _pool_tile(case, seed, i), range(case["pool"])))


def _roi(case):
    return case["roi_x"], case["roi_y"], case["roi_w"], case["roi_h"]


def _out_pixels(case, i):
    """(width, height) of the output of pool tile i."""
    w, h, _levels, _block, s, _content = _geometry(case, i)
    if case["call"] == "region":
        x, y, rw, rh = _roi(case)
        return -(-(x + rw) // s) - x // s, -(-(y + rh) // s) - y // s
    return -(-w // s), -(-h // s)


# ---- state and pass ---------------------------------------------------------

_SESSION = None


def _session():
    """The program's session: one per process, as one decode thread keeps."""
    global _SESSION
    if _SESSION is None:
        _SESSION = S.HipSession(0)
    return _SESSION


class _TensorSurface:
    """An output image inside a torch tensor of bytes."""

    def __init__(self, out, offset, width, height, fmt):
        self.device_ptr = out.data_ptr() + offset
        self.pitch_bytes = width * fmt.bytes_per_pixel
        self.byte_len = self.pitch_bytes * height


def _layout(dims, fmts):
    """256-byte aligned offsets of the outputs in one buffer, and its size."""
    offs, total = [], 0
    for (w, h), f in zip(dims, fmts):
        offs.append(total)
        total += (w * h * f.bytes_per_pixel + 255) & ~255
    return offs, total


def prepare(case, seed):
    sess = _session()
    pool = _pool(case, seed)
    call, n = case["call"], case["tiles"]
    state = {"call": call, "session": sess}
    if call in ("tile", "region"):
        cs, fmt, scale, _img = pool[0]
        state.update(data=cs, fmt=fmt, scale=scale, roi=_roi(case))
        return state
    which = [i % len(pool) for i in range(n)]
    fmts = [pool[i][1] for i in which]
    dims = [_out_pixels(case, i) for i in which]
    offs, total = _layout(dims, fmts)
    if call == "tiles":
        out = np.zeros(total, np.uint8)
        jobs = []
        for i, (w, h), f, o in zip(which, dims, fmts, offs):
            row = w * f.bytes_per_pixel
            jobs.append((pool[i][0], out[o:o + row * h], row))
        state.update(jobs=jobs, out=out, fmt=fmts[0])
        return state
    out = torch.zeros(total, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    surfaces = [_TensorSurface(out, o, w, h, f) for (w, h), f, o in zip(dims, fmts, offs)]
    plan = S.TilePlan(sess, [pool[i][0] for i in which], fmts, [pool[i][2] for i in which],
                      surfaces=surfaces)
    state.update(plan=plan, out=out)
    return state


def run(state):
    call = state["call"]
    if call == "replay":
        state["plan"].decode(S.MODE_GRAPH)
        return state["out"]
    if call == "tiles":
        S.decode_tiles_into(state["jobs"], state["fmt"], session=state["session"])
        return state["out"]
    dec = S.J2kDecoder(state["data"], state["session"])
    if call == "tile":
        return dec.decode_to_numpy(state["fmt"], state["scale"])
    return dec.decode_region_to_numpy(state["fmt"], state["roi"], state["scale"])


# ---- what is counted and compared --------------------------------------------

def work(case):
    """The coded bytes, read once, and the decoded pixels, written once.  The
    coded bytes of a region are its share of the image's area."""
    pool = _pool(case, 1)
    total = 0.0
    for i in range(case["tiles"]):
        k = i % len(pool)
        cs, fmt, _scale, img = pool[k]
        w, h = _out_pixels(case, k)
        coded = len(cs)
        if case["call"] == "region":
            coded *= case["roi_w"] * case["roi_h"] / (img.shape[0] * img.shape[1])
        # at 1/s a decode leaves out the finest levels' bands: about 1 / s^2 of the bytes
        coded /= _geometry(case, k)[4] ** 2
        total += coded + w * h * fmt.bytes_per_pixel
    return {"bytes": total, "flops": 0}


def tolerance(case):
    """Decoded samples are whole numbers, the same from every 5/3 decoder.
    9/7 is lifted in f32: against the same lifting in f64 2.8e-5 of the bytes
    of these tiles round to the neighbouring value."""
    return {"differ": 1.2e-4} if case["wavelet"] == "9/7" else "exact"


def exact(case, seed):
    """A lossless decode gives back the source pixels.  None where the output
    is not the source: 9/7, reduced resolutions, and refinement passes (the
    encoder's last bit-plane keeps only what SigProp and MagRef reach)."""
    if (case["wavelet"] == "9/7" or case["coder"] == "ht-refined" or case["scale"] != 1 or
            case["content"] == "mixed"):
        return None
    with ThreadPoolExecutor(16) as ex:
        imgs = list(ex.map(
            lambda i: _pixels(_geometry(case, i)[5], synth.tile_rng(seed, i), i,
                              case["width"], case["height"])[0], range(case["pool"])))
    imgs = [v if v.ndim == 3 else v[..., None] for v in imgs]
    if case["call"] == "tile":
        return imgs[0]
    if case["call"] == "region":
        x, y, w, h = _roi(case)
        return imgs[0][y:y + h, x:x + w]
    flat = [np.ascontiguousarray(v).view(np.uint8).reshape(-1) for v in imgs]
    step = (flat[0].size + 255) & ~255
    out = np.zeros(step * case["tiles"], np.uint8)
    for i in range(case["tiles"]):
        v = flat[i % len(flat)]
        out[i * step:i * step + v.size] = v
    return out
