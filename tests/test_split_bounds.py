"""The three bf16 pieces of csrc/split.h, restated in numpy: that they add up to the value, how large they
are, and that the error bound the GPU layer tests hold (test_gpu_split_f32.rms_bound) passes the six piece
products and fails any five of them."""

import numpy as np
import pytest

from tests.test_gpu_split_f32 import CASES, rms_bound

CUT = 2.0 ** 15


def _bf16(v):
    """Round to nearest even; the values here are finite as bf16."""
    b = np.asarray(v, np.float32).view(np.uint32)
    return ((b + 0x7FFF + ((b >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)


def pieces(v):
    v = np.asarray(v, np.float32)
    p0 = np.where(np.abs(v) < CUT, _bf16(np.where(np.abs(v) < CUT, v, 0)), (v.view(np.uint32) & 0xFFFF0000).view(np.float32))
    p1 = _bf16(v - p0)
    return p0.astype(np.float64), p1.astype(np.float64), _bf16(v - p0 - p1).astype(np.float64)


def _values(n, lo, hi, seed):
    r = np.random.default_rng(seed)
    return (np.ldexp(r.uniform(1, 2, n), r.integers(lo, hi, n)) * r.choice([-1.0, 1.0], n)).astype(np.float32)


@pytest.mark.parametrize("lo,hi", [(-100, -50), (-20, 15), (14, 17), (15, 127), (127, 128)])
def test_the_pieces_add_up_to_the_value(lo, hi):
    v = np.concatenate([_values(100000, lo, hi, 1), np.array([0x7F7F7FFF, 0x7F7F8000, 0x7F7FFFFF], np.uint32).view(np.float32)
                        if hi == 128 else np.zeros(1, np.float32)])
    p0, p1, p2 = pieces(v)
    assert np.isfinite(p0).all()
    np.testing.assert_array_equal(p0 + p1 + p2, v.astype(np.float64))
    big = np.abs(v) >= CUT
    assert np.all(np.abs(p1) <= np.abs(v.astype(np.float64)) * np.where(big, 2.0 ** -7, 2.0 ** -8))
    assert np.all(np.abs(p2) <= np.abs(v.astype(np.float64)) * np.where(big, 2.0 ** -16, 2.0 ** -17))
    # Cut off, p1 has the value's sign: an overflowing a1 b1 is the infinity of a0 b0.
    assert np.all((np.sign(p1) == np.sign(v))[big & (p1 != 0)])


def test_the_dropped_products():
    a, b = pieces(_values(1000000, -5, 5, 2)), pieces(_values(1000000, -5, 5, 3))
    rel = np.abs(a[1] * b[2] + a[2] * b[1] + a[2] * b[2]) / np.abs(sum(a) * sum(b))
    assert rel.max() <= 2.0 ** -24 * 1.01 and np.sqrt(np.mean(rel ** 2)) <= 2.0 ** -27


KS = sorted({c[1] * 4 if c[0][0] == "t" else c[1] // c[3] * {"1x1": 1, "2x2": 4}.get(c[0], 9) for c in CASES})


@pytest.mark.parametrize("k", KS)
def test_every_piece_product_is_needed(k):
    """Sums of K random products as the layer test draws them, in 64 bits: six piece products are inside
    its bound with what they drop, and a sixth missing is outside it, by a factor of two at least."""
    r = np.random.default_rng(k)
    n = max(1000, 200000 // k)
    a, b = r.standard_normal((n, k)).astype(np.float32), r.standard_normal((n, k)).astype(np.float32)
    pa, pb = pieces(a), pieces(b)
    exact, s2 = a.astype(np.float64) * b, np.sqrt(np.sum((a.astype(np.float64) * b) ** 2, 1))
    prod = {(i, j): pa[i] * pb[j] for i, j in ((0, 0), (1, 1), (1, 0), (0, 2), (0, 1), (2, 0))}

    def rms(keys):
        return np.sqrt(np.mean(((sum(prod[q] for q in keys) - exact).sum(1) / s2) ** 2))

    assert rms(prod) <= 0.25 * rms_bound(k)
    for q in prod:
        assert rms([p for p in prod if p != q]) >= 2 * rms_bound(k), (q, rms([p for p in prod if p != q]), rms_bound(k))
