"""mis_snake (csrc/codec_kernels.h) restated operation by operation in float32, its coefficients read from there: its error against 64 bits, beside that of the form it took the place of, and its ends."""
import pathlib
import re

import numpy as np
import pytest

F = np.float32
HEADER = pathlib.Path(__file__).resolve().parents[1] / "mlx-audio-swift_amd" / "csrc" / "codec_kernels.h"
BODY = re.search(r"float mis_snake\(float x, float a, float ra\) \{(.*?)\n\}", HEADER.read_text(), re.S).group(1)
C = [F(v) for v in reversed(re.findall(r"([-+]?\d\.\d+e[-+]\d+)f", BODY))]      # the highest degree stands first there


def fma(a, b, c):
    return (np.asarray(a, np.float64) * np.asarray(b, np.float64) + np.asarray(c, np.float64)).astype(F)


def snake(x, a, ra):
    """a = alpha / pi, rounded once."""
    f = fma(a, x, -np.rint((a * x).astype(F)))
    s = (f * f).astype(F)
    p = fma(s, C[5], C[4])
    for k in C[3::-1]:
        p = fma(s, p, k)
    return fma(ra, (p * s).astype(F), x)


def snake_by_sine(x, alpha, ra):
    """alpha x reduced by multiples of pi, the square of a polynomial for the sine (tests/test_codec_math_cpu.py)."""
    from test_codec_math_cpu import sin_sq_f32
    return fma(ra, sin_sq_f32((alpha * x).astype(F)), x)


def test_body():
    """The operations that snake() restates, in the kernel's words."""
    lines = [re.sub(r"\s+", " ", l.strip()) for l in BODY.strip().splitlines()]
    assert len(C) == 6 and len(lines) == 8
    assert lines[0] == "const float f = fmaf(a, x, -rintf(a * x));" and lines[1] == "const float s = f * f;"
    assert lines[2].startswith("float p = fmaf(s, ") and all(l.startswith("p = fmaf(s, p, ") for l in lines[3:7]) and lines[7] == "return fmaf(ra, p * s, x);"


@pytest.mark.parametrize("scale,bound", [(0.3, 2.5e-8), (1.0, 5e-8), (3.0, 1.15e-7), (10.0, 3.5e-7), (30.0, 1.05e-6), (100.0, 3.5e-6)])
def test_error_against_64_bits(scale, bound):
    """Rounding of a (at most 2^-24 |alpha x|, 2^-25.8 rms) times the slope of sin^2 / alpha, at most one, and that of the sum.  A product that is rounded before its
    whole number is taken off has as much again: 1.06 times the form before at three, 1.15 from ten on."""
    r = np.random.default_rng(5)
    alpha = r.uniform(0.5, 2.0, 400_000).astype(F)
    x = (r.standard_normal(400_000) * scale).astype(F)
    ra = (1.0 / (alpha.astype(np.float64) + 1e-9)).astype(F)
    a = (alpha.astype(np.float64) / np.pi).astype(F)
    exact = x.astype(np.float64) + np.sin(alpha.astype(np.float64) * x.astype(np.float64)) ** 2 / (alpha.astype(np.float64) + 1e-9)
    rms = lambda y: float(np.sqrt(np.mean((y - exact) ** 2)))
    here, before = rms(snake(x, a, ra)), rms(snake_by_sine(x, alpha, ra))
    assert here <= bound and here <= 1.05 * before, (here, before)


def test_ends():
    one = np.ones(1, F)
    assert snake(np.zeros(1, F), one, one)[0] == 0.0                      # zero padding stays zero
    assert snake(np.array([0.7], F), np.zeros(1, F), np.zeros(1, F))[0] == F(0.7)      # alpha = 1 / alpha = 0: the identity
    for n in (1.0, 2.0, 1000.0, 2.0 ** 22):                                  # whole numbers of pi: sin is zero
        assert snake(np.array([n], F), one, one)[0] == F(n)
    assert abs(snake(np.array([0.5], F), one, one)[0] - 1.5) < 2e-7                    # half of one: sin is one
    with np.errstate(invalid="ignore"):
        assert np.isnan(snake(np.array([np.inf], F), one, one)[0]) and np.isnan(snake(np.array([np.nan], F), one, one)[0])
