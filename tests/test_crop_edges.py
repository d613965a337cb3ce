"""Face crops on the GPU where the crop kernel's bands, taps and word loads can go wrong: frames whose rows start at any
address and are followed by padding, the last pixel of the last row, frames of one to a few pixels, shrinks past four
source pixels per canvas pixel, unaligned output, crops of every scale.  Byte for byte against a numpy float32 / integer
restatement of the resize (engine/preprocess/cvresize.cpp), itself checked against the golden crops on the CPU."""
import hashlib
import json
import math
from pathlib import Path

import numpy as np
import pytest

import crop_cases

GOLDEN = json.loads((Path(__file__).resolve().parent / "golden" / "crops_golden.json").read_text())
f32 = np.float32


def area_taps(ssize, dsize):
    scale = 1.0 / (dsize / ssize)
    out = []
    for d in range(dsize):
        f1 = d * scale
        f2 = f1 + scale
        cell = min(scale, ssize - f1)
        s1, s2 = math.ceil(f1), min(math.floor(f2), ssize - 1)
        s1 = min(s1, s2)
        t = []
        if s1 - f1 > 1e-3:
            t.append((s1 - 1, f32((s1 - f1) / cell)))
        t += [(s, f32(1.0 / cell)) for s in range(s1, s2)]
        if f2 - s2 > 1e-3:
            t.append((s2, f32(min(min(f2 - s2, 1.0), cell) / cell)))
        out.append(t)
    return out


def round_u8(x):
    return np.clip(np.rint(x), 0, 255).astype(np.uint8)


def resize(img, dw, dh, linear):
    """cv2.resize of uint8 [h][w][3] as the reference restates it."""
    sh, sw = img.shape[:2]
    if (sw, sh) == (dw, dh):
        return img.copy()
    sx, sy = 1.0 / (dw / sw), 1.0 / (dh / sh)
    ix, iy = int(np.rint(sx)), int(np.rint(sy))
    whole = abs(sx - ix) < np.finfo(float).eps and abs(sy - iy) < np.finfo(float).eps
    if linear and not (whole and ix == iy == 2):
        def axis(s, d, scale, clip):
            ofs, coef, one = [], [], []
            for i in range(d):
                f = f32((i + 0.5) * scale - 0.5)
                o = math.floor(f)
                f = f32(f - f32(o))
                if clip and o < 0:
                    f, o = f32(0), 0
                single = bool(one and one[-1])
                if clip and o + 1 >= s:
                    single = True
                    if o >= s - 1:
                        f, o = f32(0), s - 1
                ofs.append(o)
                one.append(single)
                coef.append((int(np.rint(f32((f32(1) - f) * f32(2048)))), int(np.rint(f32(f * f32(2048))))))
            return np.array(ofs), np.array(coef, np.int64), np.array(one)
        xo, xc, one = axis(sw, dw, sx, True)
        yo, yc, _ = axis(sh, dh, sy, False)
        a = img.astype(np.int64)
        h = np.where(one[None, :, None], a[:, xo] * 2048,
                     a[:, xo] * xc[None, :, 0, None] + a[:, np.minimum(xo + 1, sw - 1)] * xc[None, :, 1, None])
        r0, r1 = h[np.clip(yo, 0, sh - 1)] >> 4, h[np.clip(yo + 1, 0, sh - 1)] >> 4
        return ((((yc[:, 0, None, None] * r0) >> 16) + ((yc[:, 1, None, None] * r1) >> 16) + 2) >> 2).astype(np.uint8)
    if whole:
        sums = img.astype(np.int64).reshape(dh, iy, dw, ix, 3).sum((1, 3))
        return ((sums + 2) >> 2).astype(np.uint8) if ix == iy == 2 else round_u8(sums.astype(f32) * f32(1.0 / f32(ix * iy)))
    a = img.astype(f32)
    tx, ty = area_taps(sw, dw), area_taps(sh, dh)
    t = np.zeros((sh, dw, 3), f32)
    for d, taps in enumerate(tx):
        for s, w in taps:
            t[:, d] = t[:, d] + a[:, s] * w
    out = np.zeros((dh, dw, 3), f32)
    for d, taps in enumerate(ty):
        acc = None
        for s, w in taps:
            v = w * t[s]
            acc = v if acc is None else acc + v
        out[d] = acc
    return round_u8(out)


def canvas(img):
    h, w = img.shape[:2]
    scale = min(720.0 / h, 1280.0 / w)
    nh, nw = max(1, round(h * scale)), max(1, round(w * scale))
    c = np.zeros((720, 1280, 3), np.uint8)
    top, left = (720 - nh) // 2, (1280 - nw) // 2
    c[top:top + nh, left:left + nw] = resize(img, nw, nh, scale >= 1)
    return c


def crop(cv, rect):
    x, y, w, h = rect
    return resize(cv[4 * y:4 * (y + h), 4 * x:4 * (x + w)], 320, 180, False)


def test_restatement_matches_golden():
    seen = {}
    for cid, (w, h), seed, rect in crop_cases.cases():
        if w * h > 1_500_000 or cid.endswith(("#1", "#2", "#3")):
            continue
        if seed not in seen:
            seen[seed] = canvas(crop_cases.frame(w, h, seed))
        assert hashlib.sha256(crop(seen[seed], rect).tobytes()).hexdigest() == GOLDEN[cid], cid


RECTS = [(0, 0, 80, 45), (240, 135, 80, 45), (3, 5, 80, 90), (17, 30, 93, 61), (100, 40, 160, 90), (70, 39, 180, 101),
         (0, 0, 320, 180), (1, 1, 317, 179), (40, 0, 240, 180), (139, 0, 181, 180)]
# (width, height, row padding, byte offset of the frame)
FRAMES = [(1920, 1080, 0, 0), (1366, 768, 5, 1), (1000, 1000, 3, 3), (853, 479, 1, 2), (1280, 720, 0, 1), (5, 3, 0, 1),
          (1, 1, 0, 3), (2, 7, 2, 1), (641, 361, 7, 2), (5761, 3241, 2, 1), (7680, 4320, 0, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("w,h,pad,off", FRAMES)
def test_gpu_crops_any_stride_and_alignment(shv, w, h, pad, off):
    print(f"[gpu] crops of a {w}x{h} frame, {pad} bytes of row padding, at byte {off}", flush=True)
    hip = shv.Hip()
    rng = np.random.default_rng(w * 7 + h)
    img = rng.integers(0, 256, (h, w, 3), dtype=np.uint8)
    stride = 3 * w + pad
    # the buffer ends with the frame's last pixel
    buf = rng.integers(0, 256, off + (h - 1) * stride + 3 * w, dtype=np.uint8)
    for y in range(h):
        buf[off + y * stride:off + y * stride + 3 * w] = img[y].reshape(-1)
    want = [crop(c, r) for c in [canvas(img)] for r in RECTS]
    d, d_out = hip.upload(buf), hip.malloc(len(RECTS) * shv.FRAME_BYTES + 8)
    try:
        for shift in (0, 1):
            hip.memset(d_out, 0xA5, len(RECTS) * shv.FRAME_BYTES + 8)
            shv.native_crops_rgb([(d + off, w, h, stride)] * len(RECTS), RECTS, d_out + shift)
            got = hip.download(d_out, len(RECTS) * shv.FRAME_BYTES + 8, np.uint8)
            n = len(RECTS) * shv.FRAME_BYTES
            assert np.all(got[:shift] == 0xA5) and np.all(got[shift + n:] == 0xA5)
            got = got[shift:shift + n].reshape(len(RECTS), 180, 320, 3)
            for r, g, e in zip(RECTS, got, want):
                assert np.array_equal(g, e), (r, int(np.abs(g.astype(int) - e.astype(int)).max()))
    finally:
        hip.free(d)
        hip.free(d_out)


def yuv_to_rgb(Y, U, V):
    """ffmpeg's unscaled yuv420p -> rgb24 in 16-bit fixed point (engine/preprocess/color.cpp:4-11, 57-109)."""
    h, w = Y.shape
    u, v = (c.repeat(2, 0).repeat(2, 1)[:h, :w].astype(np.int64) for c in (U, V))

    def r16(f):
        return int(np.clip((f + (1 << 15)) >> 16, -32768, 32767))
    cy, vr, ub, ug, vg = (r16(c * (1 << 13)) for c in ((65536 * 255) // 219, 104597, 132201, -25675, -53279))
    y = (((Y.astype(np.int64) << 3) - r16((16 << 16) * 8)) + 32768) % 65536 - 32768
    u, v = (np.clip((c << 3) - 0x0400, -32768, 32767) for c in (u, v))
    yy = (y * cy) >> 16
    cg = np.clip(((u * ug) >> 16) + ((v * vg) >> 16), -32768, 32767)
    rgb = [yy + ((v * vr) >> 16), yy + cg, yy + ((u * ub) >> 16)]
    return np.stack([np.clip(np.clip(c, -32768, 32767), 0, 255) for c in rgb], -1).astype(np.uint8)


@pytest.mark.gpu
@pytest.mark.parametrize("w,h,pad,off", [(1920, 1080, 0, 0), (1365, 767, 3, 1), (1280, 720, 1, 3), (5, 3, 0, 1), (1, 1, 0, 0),
                                         (641, 361, 2, 2), (5761, 3241, 1, 1)])
def test_gpu_i420_crops_any_stride_and_alignment(shv, w, h, pad, off):
    print(f"[gpu] I420 crops of a {w}x{h} frame, {pad} bytes of row padding, at byte {off}", flush=True)
    hip = shv.Hip()
    rng = np.random.default_rng(w * 11 + h)
    cw, ch = (w + 1) // 2, (h + 1) // 2
    planes = [rng.integers(0, 256, s, dtype=np.uint8) for s in ((h, w), (ch, cw), (ch, cw))]
    want = [crop(c, r) for c in [canvas(yuv_to_rgb(*planes))] for r in RECTS]
    dev, args = [], []
    d_out = hip.malloc(len(RECTS) * shv.FRAME_BYTES)
    try:
        for p in planes:
            stride = p.shape[1] + pad
            buf = np.zeros(off + (p.shape[0] - 1) * stride + p.shape[1], np.uint8)
            for y in range(p.shape[0]):
                buf[off + y * stride:off + y * stride + p.shape[1]] = p[y]
            dev.append(hip.upload(buf))
            args.append((dev[-1] + off, stride))
        frame = (args[0][0], args[1][0], args[2][0], args[0][1], args[1][1], args[2][1], w, h)
        shv.native_crops_i420([frame] * len(RECTS), RECTS, d_out)
        got = hip.download(d_out, (len(RECTS), 180, 320, 3), np.uint8)
        for r, g, e in zip(RECTS, got, want):
            assert np.array_equal(g, e), (r, int(np.abs(g.astype(int) - e.astype(int)).max()))
    finally:
        for p in (*dev, d_out):
            hip.free(p)
