"""The crop kernel's word loads stay inside every plane: worked out on the CPU from the plans and the choice of kernel that
the library compiles (tests/native/crop_reach.cpp), and on the GPU the crops of I420 frames of one to a few columns, whose
chroma rows are shorter than a word, byte for byte."""
import subprocess
from pathlib import Path

import pytest

import test_crop_edges as edges

HERE = Path(__file__).resolve().parent


def test_word_loads_stay_in_their_planes(tmp_path):
    exe = tmp_path / "crop_reach"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", str(HERE / "native" / "crop_reach.cpp"), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("w,h,pad", [(1, 720, 0), (2, 3, 0), (2, 720, 0), (3, 720, 1), (3, 5, 0), (4, 3, 0), (4, 64, 1),
                                     (4, 2880, 0), (5, 4, 0), (6, 7, 0)])
def test_gpu_narrow_i420_crops(shv, w, h, pad):
    edges.test_gpu_i420_crops_any_stride_and_alignment(shv, w, h, pad, 0)
