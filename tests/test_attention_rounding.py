"""The bound behind the attention kernel's rounding of P (attention_i8.hip):
the exponent it forms in one fused step against the reference's roundings,
on the CPU; and, on the GPU, scores of every magnitude against the oracle."""
import os
import re

import numpy as np
import pytest

from helpers import f32_bits_equal, mismatch_report

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
L2E, L255, U = np.float32(1.44269504088896341), np.float32(7.99435343685885793), 2.0 ** -24


def fma(a, b, c):
    """float32 fma (the product of two float32 is exact in float64)."""
    return (a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64)).astype(np.float32)


def kap_terms():
    """(c, d) of the kernel's kap = (c + d |m|) u."""
    src = open(os.path.join(ROOT, "indecis_amd", "csrc", "attention_i8.hip")).read()
    return [float(t) for t in re.search(r"kap = \(([0-9.]+)f \+ ([0-9.]+)f \* fabsf\(m\)\) \* 0x1p-24f", src).groups()]


def test_kap_covers_every_rounding():
    """kap against the roundings counted one by one, each at its largest: in
    the exponent s and s - m (the reference's), es, the two of eb, the exponent
    itself on either side; then exp255_fast against the reference formulas
    (10 u, verified float by float on the device), two hardware exponentials
    of 2 u and the scaling by hi. |s| <= |m| + 6.3; the constants' own errors
    are the same on both sides."""
    c, d = kap_terms()
    l2e, ln2 = 1.0 / np.log(2.0), np.log(2.0)
    for m in (0.0, 1.0, 18.0, 100.0, 32768.0):
        s = m + 6.3
        exponent = l2e * (s + 6.3) + l2e * s + 2 * (l2e * m + 8) + 2 * 8
        assert exponent * ln2 + 10 + 4 + 2 <= c + d * m, m
        kap = (c + d * m) * U  # the two bounds: e^-kap times, and that hi = 1 + 2.125 kap times
        assert (1 + kap) * np.exp(-kap) <= 1 and (1 - kap) * np.exp(-kap) * (1 + 2.125 * kap) >= 1


@pytest.mark.parametrize("top", [0.01, 1.0, 8.0, 300.0, 32768.0])
def test_exponent_error_bound(top):
    """x = f32(q.k)*ks, sq and the row max m at random, scores s = x*sq
    within 6.3 of m: the kernel's exponent, kap's share of it added back,
    differs from the one that exp255_fast forms of f32(f32(x*sq) - m) by at
    most (59.3 + 4 log2 e |m|) u, and 255*exp(s - m) lies between its two
    bounds."""
    rng = np.random.default_rng(5)
    n = 400000
    m = (rng.uniform(-top, top, n)).astype(np.float32)
    sq = np.exp(rng.uniform(-12, 4, n)).astype(np.float32)
    x = ((m - rng.uniform(0, 6.3, n)) / sq).astype(np.float32)
    s = (x * sq).astype(np.float32)
    d = (np.minimum(s, m) - m).astype(np.float32)
    keep = (s <= m) & (d >= -6.3)
    m, sq, x, d = m[keep], sq[keep], x[keep], d[keep]
    ref = fma(d, np.full_like(d, L2E), np.full_like(d, L255))
    es = (sq * L2E).astype(np.float32)
    base = fma(-m, np.full_like(m, L2E), np.full_like(m, L255))
    am = np.abs(m).astype(np.float64)
    k0, k1 = kap_terms()
    kap = ((np.float32(k0) + np.float32(k1) * np.abs(m)) * np.float32(U)).astype(np.float32)
    low = (np.float32(1.4427) * kap).astype(np.float32)
    arg = fma(x, es, (base - low).astype(np.float32)).astype(np.float64)
    err, bound = np.abs(arg + low - ref), (59.3 + 4 * 1.442696 * am) * U
    assert np.all(err <= bound), (err / bound).max()
    y = np.exp2(arg)
    hi = (np.float32(1) + np.float32(2.125) * kap).astype(np.float64)
    true = 255.0 * np.exp(d.astype(np.float64))
    # 12 u: the share of the hardware exponential and of the reference formulas
    assert np.all(y * (1 + 12 * U) <= true) and np.all(y * hi * (1 - 12 * U) >= true)


@pytest.mark.gpu
@pytest.mark.parametrize("lanes", [8, 0])
@pytest.mark.parametrize("scale", [1e-3, 0.3, 6.0, 60.0, 400.0, 1e4])
def test_attend8_score_magnitudes(scale, lanes):
    """Attend8 with q and k scaled by `scale` (row maxima of the scores from
    about 1e-5 to 1e9, either side of the bound past which every score is
    formed as the reference forms it), global and windowed, against the
    oracle, bit for bit."""
    from indecis_amd import linalg
    from oracle import oracle as orc
    rng = np.random.default_rng(int(scale * 1000) + lanes)
    for n, window in ((33, -1), (300, 8), (700, -1), (261, 64)):
        q, k, v = (rng.standard_normal((n, 64)).astype(np.float32) for _ in range(3))
        q, k = q * np.float32(scale), k * np.float32(scale)
        q[n // 2] = 0
        got, want = linalg.attend8(q, k, v, window, 0.125, lanes), orc.attend8(q, k, v, window, 0.125, lanes)
        assert f32_bits_equal(got, want), (n, window, mismatch_report(got, want))


@pytest.mark.gpu
@pytest.mark.parametrize("lanes", [8, 0])
@pytest.mark.parametrize("qmax", [3.2e38, 2.9e38])
def test_attend8_query_scale_overflow(qmax, lanes):
    """Queries near the largest float with a scale of 100: the query scale
    max|q|/127*100 is finite (2.5e38 and 2.3e38), its product with log2 e is
    not (it is, for the second), and the scores are a few units (one key:
    zero), against the oracle, bit for bit."""
    from indecis_amd import linalg
    from oracle import oracle as orc
    rng = np.random.default_rng(lanes)
    for n, window in ((1, -1), (2, -1), (33, 4), (300, -1), (700, 64)):
        q, k = np.zeros((n, 64), np.float32), (3e-37 * rng.standard_normal((n, 64))).astype(np.float32)
        q[:, 0] = qmax
        q[:, 1] = np.float32(qmax) / np.float32(127) * rng.integers(1, 3, n).astype(np.float32)
        k[:, 0] = 0
        k[:, 1] *= np.float32(0.05)
        v = rng.standard_normal((n, 64)).astype(np.float32)
        got, want = linalg.attend8(q, k, v, window, 100.0, lanes), orc.attend8(q, k, v, window, 100.0, lanes)
        assert np.isfinite(want).all()
        assert f32_bits_equal(got, want), (n, window, mismatch_report(got, want))
