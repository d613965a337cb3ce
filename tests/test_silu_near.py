"""SHIELD-A's SiLU (shield-sisa_amd/csrc/silu_near.hpp) against x / (1 + exp(-x)) in 80 bits, over the whole range down to
where its result becomes -0, and at its limits (zeros, the clamp, infinities, NaN).  CPU only: the function is compiled with
stand-ins for the hardware's exp2 and reciprocal, each at every error that their 1 ulp allows.

The bounds: exp2 an ulp off its rounded value is a relative error of 1.5 x 2^-23 at most, 3 ulp of a result whose mantissa is
near 2; the residual step takes the reciprocal's error out up to its own last rounding, half an ulp: 3.5 ulp for x > -16.
Below, dl's last bit can be one ulp of d off: 4.5."""
import subprocess
from pathlib import Path

HERE = Path(__file__).resolve().parent


def test_silu_near(tmp_path):
    exe = tmp_path / "silu_near"
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-Wall", "-Wextra", "-Werror",
                    str(HERE / "native" / "silu_near.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=120).stdout.splitlines()
    assert len(out) == 1, out
    upper, lower = map(float, out[0].split())
    assert upper <= 3.5 and lower <= 4.5, out[0]
