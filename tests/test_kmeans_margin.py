"""The k-means screen's margin against its own arithmetic (no GPU needed).

The screen computes a = x.c - |c|^2 / 2 from two fp16 terms of each value and
keeps an index in the low 4 bits; whatever its distance from the exact a, the
margin M of hml_k_kmeans.hip has to cover it twice.  Here the screen is
restated in numpy, one rounding per step, on values whose terms round worst
(just off the middle between two fp16 numbers), on random ones and on small
ones, where fp16 loses its normal range; the margin's factors are read from
the kernel's source."""
import os
import re

import numpy as np
import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hiperml_amd", "csrc",
                   "hml_k_kmeans.hip")
U = 2.0 ** -24


def factors(ks):
    """The source's factors of |x|^2 and |c|^2 and its constant for ks
    k-steps, in units of u."""
    text = open(SRC).read()
    a, b, c, d = (int(v) for v in re.search(
        r"kMx = \((\d+) \* KS \+ (\d+)\) \* kU, kMc = \((\d+) \* KS \+ (\d+)\) \* kU;", text).groups())
    e, = re.search(r"const float m0 = .*, (\d+) \* kU\);", text).groups()
    return a * ks + b, c * ks + d, int(e)


def terms(v):
    hi = v.astype(np.float16)
    lo = (v - hi.astype(np.float32)).astype(np.float16)
    return hi.astype(np.float32), lo.astype(np.float32)


def screen(x, c):
    """a~ of rows x (n, D) and centroids c (n, D), pairwise, float32."""
    (xh, xl), (ch, cl) = terms(x), terms(c)
    n2 = np.zeros(len(x), np.float32)
    for d in range(x.shape[1]):
        n2 = (n2.astype(np.float64) + c[:, d].astype(np.float64) ** 2).astype(np.float32)
    acc = np.float32(-0.5) * n2
    D = x.shape[1]
    for s in range(0, D, 16):
        for p, q in ((cl, xh), (ch, xl), (ch, xh)):
            for d in range(s, min(D, s + 16)):
                acc = (acc.astype(np.float64) + p[:, d].astype(np.float64) * q[:, d]).astype(np.float32)
    worst = (acc.view(np.uint32) & ~np.uint32(15))
    return acc, worst.view(np.float32), (worst | np.uint32(15)).view(np.float32)


def worst_rounding(rng, n, D):
    """Values whose fp16 terms leave the largest residuals, over three binades."""
    base = 1.0 + rng.integers(0, 1024, (n, D)) * 2.0 ** -10
    off = 2.0 ** -11 * (1 - 2.0 ** -12 * rng.integers(1, 3, (n, D)))
    v = (base + off) * 2.0 ** -rng.integers(0, 3, (n, D))
    return (v * rng.choice([-1, 1], (n, D))).astype(np.float32)


@pytest.mark.parametrize("D", [1, 2, 15, 16, 17, 32, 47, 64])
def test_margin_covers_the_screen(D):
    rng = np.random.default_rng(D)
    n, ks = 4000, (D + 15) // 16
    mx, mc, ma = factors(ks)
    uni = lambda s: (s * rng.uniform(-1, 1, (n, D))).astype(np.float32)
    same = np.abs(worst_rounding(rng, n, D))  # products of one sign: no cancelling of errors
    for x, c in ((worst_rounding(rng, n, D), worst_rounding(rng, n, D)), (same, same[::-1].copy()),
                 (uni(1), uni(1)), (uni(4000), uni(1)), (uni(1), uni(4000)), (uni(1e-3), uni(1)),
                 (uni(1e-4), uni(1e-4)), (uni(1e-7), uni(1e-7)), (uni(1), uni(1e-6))):
        x64, c64 = x.astype(np.float64), c.astype(np.float64)
        a = (x64 * c64).sum(1) - 0.5 * (c64 ** 2).sum(1)
        X, C = np.linalg.norm(x64, axis=1), np.linalg.norm(c64, axis=1)
        half = 0.5 * U * (mx * X ** 2 + mc * C ** 2 + ma)
        for got in screen(x, c):
            err = np.abs(got.astype(np.float64) - a)
            assert (err <= half).all(), (err / half).max()
