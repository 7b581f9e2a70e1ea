"""The measured cases: fused chains as a user's program runs them on one GPU.

A case names one public chain of `fusedkernellibrary_amd`, its sizes and its options.  listed() holds twelve of them, draw() gives
more of the same ranges, prepare() makes what a program has in hand before the call (frames in device memory, the regions that a
detector asked for, the tensors that receive the result), run() is one call of the chain.

Chains whose arguments change from frame to frame (regions, matrices, the ring slot) are called directly.  Chains that run with the
same buffers and values again and again can be bound once (`bound`: the library's `defer=True`, its form for launch loops).
Rows are tight, as torch allocates them, or start at multiples of 256 bytes (`row_align`), as decoders and pitched allocations have them.
Every result is specified bit for bit (the arithmetic is IEEE float32 in a fixed order, without contraction), so outputs are compared exactly.
"""
import math

import torch

import fusedkernellibrary_amd as fk

YUV_FORMATS = {"NV12": fk.NV12, "NV21": fk.NV21, "P010": fk.P010, "P210": fk.P210, "Y210": fk.Y210, "UYVY": fk.UYVY}
WIDE_FORMATS = ("P010", "P210", "Y210")  # 16-bit samples
ASPECTS = {"preserve": fk.PRESERVE_AR, "ignore": fk.IGNORE_AR, "preserve_even": fk.PRESERVE_AR_RN_EVEN, "preserve_left": fk.PRESERVE_AR_LEFT}
MATRICES = {"full601": (fk.RANGE_FULL, fk.BT601), "full709": (fk.RANGE_FULL, fk.BT709), "limited709": (fk.RANGE_LIMITED, fk.BT709),
            "full2020": (fk.RANGE_FULL, fk.BT2020)}
DEPTHS = list(fk.CHAIN_DEPTHS)
RINGS = [2, 3, 4, 8, 16]


def listed():
    return [
        # a detector's five small regions -> one 60x60 batch: the README's example at its own sizes, all launch and host latency
        dict(name="rois_5_to_60x60", chain="rois", w=1920, h=1080, row_align=1, n=5, side_min=11, side_max=70, dst_w=60, dst_h=60, aspect="preserve", bound=False),
        # five large regions of a 4K frame -> full-HD float images: the same pipeline where bandwidth counts
        dict(name="rois_5_to_1080p", chain="rois", w=3840, h=2160, row_align=1, n=5, side_min=768, side_max=1024, dst_w=1920, dst_h=1080, aspect="preserve", bound=False),
        # a busy frame of an odd-sized camera (rows of 4098 bytes), twenty-three regions of any size -> 299x299, anchored left
        dict(name="rois_23_ragged", chain="rois", w=1366, h=768, row_align=1, n=23, side_min=31, side_max=477, dst_w=299, dst_h=299, aspect="preserve_left", bound=False),
        # fifty images, one crop of each -> normalised planar 224x224: a classifier's input batch
        dict(name="batch50_to_224_planes", chain="batch", w=1920, h=1080, row_align=1, n=50, side_min=16, side_max=512, dst_w=224, dst_h=224, bound=False),
        # thirty-two tiles of a 4K frame seen at 1280x720, without the resized frame in memory: sliding-window inference
        dict(name="tiles32_of_720p", chain="tiles", w=3840, h=2160, row_align=1, rs_w=1280, rs_h=720, n=32, tile=128, bound=False),
        # sixteen element-wise operations over a 4K float image in one launch: vertical fusion
        dict(name="chain16_4k", chain="chain", w=3840, h=2160, depth=16, bound=True),
        # a decoder's 4K surface -> packed RGB bytes
        dict(name="nv12_4k_to_rgb", chain="decode", w=3840, h=2160, row_align=1, format="NV12", matrix="full709", alpha=False, float_out=False, bound=True),
        # unpacked pixels -> an encoder's full-HD surface
        dict(name="nv12_1080p_encode", chain="encode", w=1920, h=1080, row_align=1, format="NV12", bound=True),
        # a region of a decoder's 4K surface -> RGB -> 1280x720 normalised planes: a network's input straight from video
        dict(name="nv12_crop_to_720p_planes", chain="planes", w=3840, h=2160, row_align=1, format="NV12", matrix="full709", crop_w=1920, crop_h=1080, dst_w=1280, dst_h=720,
             bound=False),
        # a 4K frame rotated by a few degrees: stabilisation
        dict(name="rotate_4k", chain="warp", w=3840, h=2160, row_align=1, kind="affine", dst_w=3840, dst_h=2160, degrees=5.0, scale=1.0, bound=False),
        # one new frame into a ring of eight full-HD frames, kept as planes ordered by age: temporal models
        dict(name="ring8_1080p", chain="ring", w=1920, h=1080, row_align=1, batch=8, newest_first=True, bound=False),
        # four products of one 8K x 8K image in one launch: divergent horizontal fusion, the largest
        dict(name="divergent4_8k", chain="divergent", w=8192, h=8192, row_align=1, rs_w=512, rs_h=512, crop_w=1024, crop_h=1024, bound=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _frame(rng, lo, hi, even=False):
    """Frame sizes from `lo` to `hi` pixels wide, landscape ratios; `even` for the YUV formats."""
    w = _log_int(rng, lo, hi)
    h = max(8, int(w * rng.uniform(0.5, 0.75)))
    return (w & ~1, h & ~1) if even else (w, h)


def _layout(rng):
    return dict(row_align=rng.choice([1, 1, 256]), bound=rng.random() < 0.4)


def draw(rng):
    chain = rng.choice(["rois", "rois", "batch", "tiles", "chain", "decode", "encode", "planes", "warp", "ring", "divergent"])
    c = dict(chain=chain)
    if chain == "rois":
        w, h = _frame(rng, 320, 3840)
        lo = _log_int(rng, 8, h // 4)
        dst_w = _log_int(rng, 32, 1920)
        dst_h = _log_int(rng, 32, 1080)
        most = max(1, min(128, 10_400_000 // (dst_w * dst_h)))
        c.update(w=w, h=h, n=_log_int(rng, 1, most), side_min=lo, side_max=_log_int(rng, lo, h), dst_w=dst_w, dst_h=dst_h, aspect=rng.choice(sorted(ASPECTS)), **_layout(rng))
    elif chain == "batch":
        w, h = _frame(rng, 256, 1920)
        lo = _log_int(rng, 8, h // 4)
        side = _log_int(rng, 64, 512)
        c.update(w=w, h=h, n=_log_int(rng, 1, 64), side_min=lo, side_max=_log_int(rng, lo, min(h, 512)), dst_w=side, dst_h=rng.choice([side, max(48, side * 3 // 4)]),
                 **_layout(rng))
    elif chain == "tiles":
        w, h = _frame(rng, 640, 3840)
        factor = rng.uniform(0.7, 4.0)
        rs_w, rs_h = int(w / factor), int(h / factor)
        tile = _log_int(rng, 48, min(384, rs_h))
        c.update(w=w, h=h, rs_w=rs_w, rs_h=rs_h, n=_log_int(rng, 1, 64), tile=tile, **_layout(rng))
    elif chain == "chain":
        w, h = _frame(rng, 64, 3840)
        c.update(w=w, h=h, depth=rng.choice(DEPTHS), bound=rng.random() < 0.7)
    elif chain in ("decode", "encode"):
        w, h = _frame(rng, 160, 3840, even=True)
        c.update(w=w, h=h, format=rng.choice(sorted(YUV_FORMATS)), **_layout(rng))
        if chain == "decode":
            c.update(matrix=rng.choice(sorted(MATRICES)), alpha=rng.random() < 0.3, float_out=rng.random() < 0.4)
    elif chain == "planes":
        w, h = _frame(rng, 640, 3840, even=True)
        cw = _log_int(rng, 160, w)
        ch = max(16, min(h, int(cw * rng.uniform(0.5, 1.0))))
        dw = _log_int(rng, 160, 1920)
        c.update(w=w, h=h, format=rng.choice(sorted(YUV_FORMATS)), matrix=rng.choice(sorted(MATRICES)), crop_w=cw, crop_h=ch, dst_w=dw,
                 dst_h=max(16, int(dw * rng.uniform(0.5, 1.0))), **_layout(rng))
    elif chain == "warp":
        w, h = _frame(rng, 320, 3840)
        scale = math.exp(rng.uniform(math.log(0.5), math.log(2.0)))
        c.update(w=w, h=h, kind=rng.choice(["affine", "perspective"]), dst_w=max(64, min(3840, int(w / scale))), dst_h=max(64, min(2160, int(h / scale))),
                 degrees=rng.uniform(-20.0, 20.0), scale=scale, **_layout(rng))
    elif chain == "ring":
        w, h = _frame(rng, 160, 1920)
        batch = rng.choice(RINGS)
        if batch == 16 and w > 1280:
            batch = 8
        c.update(w=w, h=h, batch=batch, newest_first=rng.random() < 0.5, row_align=rng.choice([1, 256]), bound=False)
    else:
        w, h = _frame(rng, 256, 8192)
        c.update(w=w, h=h, rs_w=_log_int(rng, 64, w // 2), rs_h=_log_int(rng, 64, h // 2), crop_w=_log_int(rng, 32, w // 2), crop_h=_log_int(rng, 32, h // 2), **_layout(rng))
    return c


# ---- inputs ----------------------------------------------------------------------------------------------------------

class _Maker:
    """Inputs from a seed, made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)
        self.cpu = torch.Generator()
        self.cpu.manual_seed(seed)

    def ints(self, lo, hi, n):
        """n whole numbers from lo to hi, both included."""
        return torch.randint(lo, hi + 1, (n,), generator=self.cpu).tolist()

    def rows(self, h, row, dtype, row_align):
        """A (h, *row) tensor whose rows are tight or start at multiples of `row_align` bytes."""
        size = torch.empty((), dtype=dtype).element_size()
        width = math.prod(row)
        step = -(-width * size // row_align) * row_align // size if row_align > 1 else width
        flat = torch.empty((h, step), dtype=dtype, device="cuda")
        return flat[:, :width].unflatten(1, row) if len(row) > 1 else flat[:, :width]

    def picture(self, h, w, cn, row_align=1):
        """A picture of bytes: smooth shapes over the whole range (dark and bright areas clip) and sensor noise."""
        low = torch.rand((1, cn, max(2, h // 120), max(2, w // 120)), generator=self.g, device="cuda") * 300.0 - 22.0
        out = self.rows(h, (w, cn), torch.uint8, row_align)
        step = max(1, (1 << 24) // (w * cn))  # in bands, so that the largest pictures need little memory beside themselves
        smooth = torch.nn.functional.interpolate(low, size=(min(h, 1080), min(w, 1920)), mode="bilinear", align_corners=True)[0].permute(1, 2, 0)
        ys = torch.arange(h, device="cuda") * smooth.shape[0] // h
        xs = torch.arange(w, device="cuda") * smooth.shape[1] // w
        for y in range(0, h, step):
            band = smooth[ys[y:y + step]][:, xs]
            noise = torch.randint(-8, 9, band.shape, generator=self.g, device="cuda", dtype=torch.int8)
            out[y:y + step] = (band + noise).clamp_(0, 255).to(torch.uint8)
        return out

    def samples(self, h, width, wide, row_align):
        """Rows of raw samples: bytes, or 10-bit samples in the high bits of 16."""
        if not wide:
            out = self.rows(h, (width,), torch.uint8, row_align)
            out.copy_(self.picture(h, width, 1)[:, :, 0])
        else:
            out = self.rows(h, (width,), torch.int16, row_align)
            fine = torch.randint(0, 4, (h, width), generator=self.g, device="cuda", dtype=torch.int32)
            out.copy_((((self.picture(h, width, 1)[:, :, 0].to(torch.int32) << 2) | fine) << 6).to(torch.int16))
        return out

    def regions(self, n, w, h, lo_w, hi_w, lo_h=None, hi_h=None):
        """n rectangles inside a w x h frame, sides between the limits."""
        lo_h, hi_h = (lo_w if lo_h is None else lo_h), (hi_w if hi_h is None else hi_h)
        ws, hs = self.ints(min(lo_w, w), min(hi_w, w), n), self.ints(min(lo_h, h), min(hi_h, h), n)
        return [(self.ints(0, w - rw, 1)[0], self.ints(0, h - rh, 1)[0], rw, rh) for rw, rh in zip(ws, hs)]


def _raw_shape(fmt, w, h):
    """(rows, elements per row) of a raw image."""
    if fmt in ("NV12", "NV21", "P010"):
        return h + h // 2, w
    if fmt == "P210":
        return 2 * h, w
    return h, 2 * w


def _matrix(c):
    """Destination -> source: a rotation about the centres with a change of scale, and a slight tilt for the perspective kind."""
    a = math.radians(c["degrees"])
    s = c["scale"]
    m = [[s * math.cos(a), -s * math.sin(a), 0.0], [s * math.sin(a), s * math.cos(a), 0.0]]
    for row, half in zip(m, (c["w"] / 2, c["h"] / 2)):
        row[2] = half - row[0] * c["dst_w"] / 2 - row[1] * c["dst_h"] / 2
    if c["kind"] == "affine":
        return fk.WARP_AFFINE, m
    return fk.WARP_PERSPECTIVE, m + [[0.04 / c["dst_w"], 0.02 / c["dst_h"], 1.0]]


def prepare(case, seed):
    c, m = case, _Maker(seed)
    chain = c["chain"]
    w, h = c["w"], c["h"]
    align = c.get("row_align", 1)
    if chain == "rois":
        frame = m.picture(h, w, 3, align)
        rects = m.regions(c["n"], w, h, c["side_min"], c["side_max"])
        out = torch.empty((c["n"], c["dst_h"], c["dst_w"], 3), device="cuda")
        call, args, result = fk.crop_resize_muls_bgr_tensor, (frame, rects, out, ASPECTS[c["aspect"]], (0, 0, 0), (1.4,) * 3, (0.5,) * 3, (255.,) * 3), out
    elif chain == "batch":
        frames = [m.picture(h, w, 3, align) for _ in range(c["n"])]
        rects = m.regions(c["n"], w, h, c["side_min"], c["side_max"])
        out = torch.empty((c["n"], 3, c["dst_h"], c["dst_w"]), device="cuda")
        call, args, result = fk.batch_crop_resize_norm_split, (frames, rects, out, (255.,) * 3, (.485, .456, .406), (.229, .224, .225)), out
    elif chain == "tiles":
        frame = m.picture(h, w, 3, align)
        rects = m.regions(c["n"], c["rs_w"], c["rs_h"], c["tile"], c["tile"])
        out = torch.empty((c["n"], c["tile"], c["tile"], 3), device="cuda")
        call, args, result = fk.resize_crop_tiles, (frame, (c["rs_w"], c["rs_h"]), rects, out, (1 / 255.,) * 3), out
    elif chain == "chain":
        src = torch.rand((h, w, 3), generator=m.g, device="cuda")
        out = torch.empty_like(src)
        call, args, result = fk.muladd_chain_f32c3, (src, out, c["depth"], 1.0001, 1e-4), out
    elif chain == "decode":
        rows, width = _raw_shape(c["format"], w, h)
        wide = c["format"] in WIDE_FORMATS
        raw = m.samples(rows, width, wide, align)
        dtype = torch.float32 if c["float_out"] else torch.int16 if wide else torch.uint8
        out = torch.empty((h, w, 4 if c["alpha"] else 3), dtype=dtype, device="cuda")
        call, args, result = fk.yuv_to_rgb, (YUV_FORMATS[c["format"]], *MATRICES[c["matrix"]], raw, out), out
    elif chain == "encode":
        rows, width = _raw_shape(c["format"], w, h)
        wide = c["format"] in WIDE_FORMATS
        pixels = m.samples(h, 3 * w, wide, 1).unflatten(1, (w, 3))
        out = m.rows(rows, (width,), torch.int16 if wide else torch.uint8, align)
        call, args, result = fk.write_yuv, (YUV_FORMATS[c["format"]], pixels, out), out
    elif chain == "planes":
        rows, width = _raw_shape(c["format"], w, h)
        raw = m.samples(rows, width, c["format"] in WIDE_FORMATS, align)
        crop = m.regions(1, w, h, c["crop_w"], c["crop_w"], c["crop_h"], c["crop_h"])[0]
        out = torch.empty((3, c["dst_h"], c["dst_w"]), device="cuda")
        top = 65535.0 if c["format"] in WIDE_FORMATS else 255.0
        call, args, result = fk.yuv_crop_resize_norm_split, (YUV_FORMATS[c["format"]], *MATRICES[c["matrix"]], raw, (w, h), crop, out, top), out
    elif chain == "warp":
        src = m.picture(h, w, 3, align)
        out = torch.empty((c["dst_h"], c["dst_w"], 3), device="cuda")
        kind, matrix = _matrix(c)
        call, args, result = fk.warp_u8c3_f32c3, (kind, matrix, src, out), out
    elif chain == "ring":
        frame = m.picture(h, w, 3, align)
        ring = torch.rand((c["batch"], 3, h, w), generator=m.g, device="cuda")
        return {"ring": ring, "tensor": torch.empty_like(ring), "frame": frame, "next": 0, "newest_first": int(c["newest_first"])}
    else:
        src = m.picture(h, w, 4, align)
        rect = m.regions(1, w, h, c["crop_w"], c["crop_w"], c["crop_h"], c["crop_h"])[0]
        result = [torch.empty((h, w), dtype=torch.uint8, device="cuda"), torch.empty((c["rs_h"], c["rs_w"], 4), device="cuda"),
                  torch.empty((c["crop_h"], c["crop_w"], 4), dtype=torch.uint8, device="cuda"), torch.empty((h, w, 3), device="cuda")]
        call, args = fk.divergent4_u8c4, (src, result[0], result[1], 1 / 255., rect, 2, result[2], 0.5, result[3])
    state = {"call": call, "args": args, "out": result, "bound": None}
    if c.get("bound"):
        state["bound"] = call(*args, defer=True)
    return state


def run(state):
    if "ring" in state:
        s = state
        s["next"] = fk.circular_tensor_update_u8c3_split_f32(s["frame"], 1 / 255., s["tensor"], s["ring"], s["next"], s["newest_first"])
        return [s["tensor"], s["ring"]]
    if state["bound"] is not None:
        state["bound"]()
    else:
        state["call"](*state["args"])
    return state["out"]


# ---- what a pass cannot do without -----------------------------------------------------------------------------------

def _raw_bytes(fmt, w, h):
    """Bytes of a w x h window of a raw image."""
    if fmt in ("NV12", "NV21"):
        return w * h * 3 // 2
    if fmt == "P010":
        return w * h * 3
    return w * h * (2 if fmt == "UYVY" else 4)


def _taken(crop_w, crop_h, dst_w, dst_h):
    """Share of a window's pixels that a bilinear resize reads: all of them up to a factor of two per axis, then two per output."""
    return min(1.0, 2.0 * dst_w / crop_w) * min(1.0, 2.0 * dst_h / crop_h)


def work(case):
    c, w, h = case, case["w"], case["h"]
    chain = c["chain"]
    if chain in ("rois", "batch"):
        side = (c["side_min"] + c["side_max"]) / 2
        px = c["n"] * c["dst_w"] * c["dst_h"]
        crop_w, crop_h = min(side, w), min(side, h)
        return {"bytes": int(px * 12 + c["n"] * crop_w * crop_h * 3 * _taken(crop_w, crop_h, c["dst_w"], c["dst_h"])), "flops": px * 3 * 10}
    if chain == "tiles":
        px = c["n"] * c["tile"] ** 2
        fx, fy = w / c["rs_w"], h / c["rs_h"]
        src = c["n"] * (c["tile"] * fx) * (c["tile"] * fy) * _taken(fx, fy, 1, 1)
        return {"bytes": int(px * 12 + min(src, w * h) * 3), "flops": px * 3 * 8}
    if chain == "chain":
        return {"bytes": w * h * 24, "flops": w * h * 3 * c["depth"]}
    if chain == "decode":
        px = (4 if c["alpha"] else 3) * (4 if c["float_out"] else 2 if c["format"] in WIDE_FORMATS else 1)
        return {"bytes": _raw_bytes(c["format"], w, h) + w * h * px, "flops": w * h * 12}
    if chain == "encode":
        return {"bytes": w * h * 3 * (2 if c["format"] in WIDE_FORMATS else 1) + _raw_bytes(c["format"], w, h), "flops": 0}
    if chain == "planes":
        px = c["dst_w"] * c["dst_h"]
        share = _taken(c["crop_w"], c["crop_h"], c["dst_w"], c["dst_h"])
        return {"bytes": int(px * 12 + _raw_bytes(c["format"], c["crop_w"], c["crop_h"]) * share), "flops": px * 3 * 8 + int(c["crop_w"] * c["crop_h"] * share) * 12}
    if chain == "warp":
        px = c["dst_w"] * c["dst_h"]
        covered = min(w * h, px * c["scale"] ** 2) * _taken(c["scale"], c["scale"], 1, 1)
        return {"bytes": int(px * 12 + covered * 3), "flops": px * 40}
    if chain == "ring":
        px, b = w * h, c["batch"]
        return {"bytes": px * 3 + px * 12 * 2 + (b - 1) * px * 12 * 2, "flops": px * 3}
    # the image once, and the four products
    px, small, crop = w * h, c["rs_w"] * c["rs_h"], c["crop_w"] * c["crop_h"]
    return {"bytes": px * 4 + px + small * 16 + crop * 4 + px * 12, "flops": px * 8 + small * 36 + crop * 4}


def tolerance(case):
    return "exact"
