"""The bf16 quantiser's division: one remainder correction gives the correctly rounded fp32 quotient.

Exact integer arithmetic over all 8-bit significands of x and of the block's maximum (the scale is the fp32 quotient
max/448), for the correctly rounded reciprocal of the scale and both of its neighbours: the kernel's reciprocal, the
hardware's refined by one Newton step, is one of the three.  Exponents do not matter: every operation scales with them as
long as nothing leaves the normal range, and where something does the code is a zero either way.
"""
from fractions import Fraction

import numpy as np
import pytest
import torch
import importlib

inputs = importlib.import_module("amd-developer-challenge-2025_amd.inputs")


def rn(x):
    """Fraction -> nearest fp32 value (24-bit significand, ties to even), unbounded exponent."""
    if x == 0:
        return Fraction(0)
    n, d = abs(x.numerator), x.denominator
    e = n.bit_length() - d.bit_length() - 24
    scaled = Fraction(n, d) / (Fraction(2) ** e)             # in (2^23, 2^25)
    if scaled >= 1 << 24:
        e += 1
        scaled /= 2
    v = Fraction(round(scaled)) * Fraction(2) ** e           # round(): ties to even
    return v if x > 0 else -v


def ulp(x):
    e = x.numerator.bit_length() - x.denominator.bit_length()
    if Fraction(2) ** e > x:
        e -= 1
    return Fraction(2) ** (e - 23)


def one_step(x, s, y):
    q = rn(x * y)
    r = rn(s * q - x)
    return rn(q - r * y)


@pytest.mark.parametrize("maxima", [range(128 + 16 * i, 144 + 16 * i) for i in range(8)] + [None])
def test_one_correction_is_exact_for_bf16(maxima):
    scales = [rn(Fraction(a, 448)) for a in maxima] if maxima is not None else [Fraction(float(np.float32(1e-12)))]
    for s in scales:
        y0 = rn(1 / s)
        for x in range(128, 256):
            want = rn(x / s)
            for y in (y0 - ulp(y0), y0, y0 + ulp(y0)):
                assert one_step(Fraction(x), s, y) == want, (float(s), x)


def _every_pair(exponent):
    """Every (maximum, x) pair of significands at ten exponent distances, both signs, and -0; the rows of distance `gap` are
    scaled by 2^(7 gap + exponent)."""
    sig = torch.arange(128, 256, dtype=torch.float32)
    rows = []
    for gap in range(10):
        for a in sig:
            x = sig * 2.0 ** -gap
            x = torch.where(x > a, x / 2, x)
            x = torch.where(torch.arange(128) % 2 == 0, x, -x)
            lo, hi = x.clone(), x.clone()
            lo[0], hi[127] = a, -a                            # both halves hold the maximum; together they hold every x
            lo[1 + gap] = -0.0
            rows.append(torch.cat([lo, hi]) * 2.0 ** (7 * gap + exponent))
    return torch.stack(rows).to(torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("exponent", [-40, -30])
def test_every_pair_of_bf16_significands(exponent):
    """The CPU quantiser's bytes.  At -30 every scale is max / 448, also at distance 0, where x is within a factor of two of the
    maximum; at -40 the rows of distance 0 have the smallest scale, 1e-12."""
    quant = importlib.import_module("amd-developer-challenge-2025_amd.quant")
    x = _every_pair(exponent)
    q, s = quant.quantize_a(x.cuda())
    rq, rs = inputs.quantize_a(x.float())
    least = torch.tensor(1e-12, dtype=torch.float32)
    assert bool((rs[:128] == least).all() if exponent == -40 else (rs > least).all()) and bool((rs[128:] > least).all())
    assert torch.equal(s.cpu(), rs)
    assert torch.equal(q.cpu().view(torch.uint8), rq.view(torch.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows", [1, 2, 3, 5, 15, 17, 31, 33, 63, 65, 127, 129, 250, 1023, 4099])
def test_rows_of_any_count(rows, dtype):
    """Rows of the output that start and end on any byte: pieces of the last chunk, and the tiles of 32 and 64 rows."""
    quant = importlib.import_module("amd-developer-challenge-2025_amd.quant")
    for k in (128, 1536):
        x = torch.randn(rows, k, generator=torch.Generator().manual_seed(rows)).to(dtype)
        q, s = quant.quantize_a(x.cuda())
        rq, rs = inputs.quantize_a(x.float())
        assert torch.equal(s.cpu(), rs) and torch.equal(q.cpu().view(torch.uint8), rq.view(torch.uint8))
        q, s = quant.quantize_b(x.cuda())
        rq, rs = inputs.quantize_b(x.float())
        assert torch.equal(s.cpu(), rs) and torch.equal(q.cpu().view(torch.uint8), rq.view(torch.uint8))
