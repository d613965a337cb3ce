"""The wide pointwise GEMM reads no weight outside its row: on the CPU the lane offsets that the kernel compiles
(tests/native/gemm_reach.cpp), on the GPU the shortest rows (K 8 to 24, fewer than a K step of 32) and the automatic choice
for them, bitwise against the direct kernel.  Beside it, both sides of its groups of two or four column tiles."""
import subprocess
from pathlib import Path

import pytest

import test_gemm_wide as wide

HERE = Path(__file__).resolve().parent


def test_weight_reads_stay_in_their_row(tmp_path):
    exe = tmp_path / "gemm_reach"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", str(HERE / "native" / "gemm_reach.cpp"), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(65, 4, 8), (2049, 176, 8), (130, 180, 16), (2050, 324, 24), (64, 192, 40)])
@pytest.mark.parametrize("mode", ["fp16", "bf16"])
def test_short_rows(shv, mode, M, N, K):
    wide.test_wide_gemm_equals_direct(shv, mode, M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("N", [192, 196, 324, 960])   # 12 column tiles in groups of four, 13, 21 (odd) and 60 in groups of two
@pytest.mark.parametrize("mode,K", [("fp16", 184), ("fp16", 192), ("bf16", 104), ("bf16", 128)])
def test_groups_of_two_or_four_tiles(shv, mode, N, K):
    wide.test_wide_gemm_equals_direct(shv, mode, 2113, N, K)
