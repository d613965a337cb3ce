"""How a call's crops are split into bands and column chunks (crop_split, shield-sisa_amd/csrc/crop_plan.hpp): few crops over
many workgroups (on the CPU, tests/native/crop_split.cpp), and on the GPU the bytes of every split: the crop counts where the
rule changes, frames of every kernel (1 to 8 source pixels per axis unrolled, more and narrow frames pixel by pixel), frames
under letterbox bars on the patch's sides or all over it, and all of them in one call."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

import test_crop_edges as edges

HERE = Path(__file__).resolve().parent
# portrait (bars left and right), wide (bars above and below), a few columns, scales of 1 to 10, enlarged
FRAMES = [(720, 1280), (405, 720), (1280, 200), (3, 400), (1920, 1080), (3840, 2161), (5120, 2880), (6400, 3600), (7000, 4000),
          (8192, 4608), (12000, 900), (640, 362), (2, 3)]
RECTS = [(0, 0, 80, 45), (240, 135, 80, 45), (120, 60, 101, 57), (0, 0, 320, 180), (77, 3, 166, 93), (100, 40, 160, 90)]


def test_few_crops_fill_the_device(tmp_path):
    exe = tmp_path / "crop_split"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", str(HERE / "native" / "crop_split.cpp"), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


class Frames:
    """Frames on the device with their canvases."""

    def __init__(self, shv, i420):
        self.shv, self.i420, self.hip, self.dev, self.args, self.canvas = shv, i420, shv.Hip(), [], [], []
        for w, h in FRAMES:
            rng = np.random.default_rng(w * 13 + h)
            cw, ch = (w + 1) // 2, (h + 1) // 2
            shapes = ((h, w), (ch, cw), (ch, cw)) if i420 else ((h, w, 3),)
            planes = [rng.integers(0, 256, s, dtype=np.uint8) for s in shapes]
            d = [self.hip.upload(p) for p in planes]
            self.dev += d
            self.args.append((*d, w, cw, cw, w, h) if i420 else (d[0], w, h, 3 * w))
            self.canvas.append(edges.canvas(edges.yuv_to_rgb(*planes) if i420 else planes[0]))

    def check(self, which, rects):
        n = len(which)
        d_out = self.hip.malloc(n * self.shv.FRAME_BYTES)
        try:
            self.hip.memset(d_out, 0xA5, n * self.shv.FRAME_BYTES)
            crops = self.shv.native_crops_i420 if self.i420 else self.shv.native_crops_rgb
            crops([self.args[f] for f in which], rects, d_out)
            got = self.hip.download(d_out, (n, 180, 320, 3), np.uint8)
        finally:
            self.hip.free(d_out)
        for f, r, g in zip(which, rects, got):
            assert np.array_equal(g, edges.crop(self.canvas[f], r)), (FRAMES[f], r, n)


@pytest.mark.gpu
@pytest.mark.parametrize("i420", [False, True], ids=["rgb", "i420"])
def test_gpu_crops_in_every_split(shv, i420):
    fr = Frames(shv, i420)
    try:
        for n in (1, 2, 3, 4, 5, 8, 9, 16, 17):
            print(f"[gpu] {n} crops of every frame, I420 {i420}", flush=True)
            for f in range(len(FRAMES)):
                fr.check([f] * n, [RECTS[(i + f) % len(RECTS)] for i in range(n)])
        every = [(f, r) for f in range(len(FRAMES)) for r in RECTS]
        print(f"[gpu] {len(every)} crops of all frames, I420 {i420}", flush=True)
        fr.check([f for f, _ in every], [r for _, r in every])
    finally:
        for d in fr.dev:
            fr.hip.free(d)
