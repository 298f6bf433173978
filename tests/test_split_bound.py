"""The arithmetic behind float products on the bf16 matrix cores: a float as
three bf16, each rounded to nearest, and what the six largest of the nine
products leave out."""

from __future__ import annotations

import numpy as np


def _nearest_bf16(x):
    bits = x.view(np.uint32).astype(np.uint64)
    return ((bits + 0x7FFF + ((bits >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)


def _parts(x):
    h = _nearest_bf16(x)
    m = _nearest_bf16(x - h)
    low = (x - h) - m
    return h, m, low


def test_three_parts_are_exact_and_small():
    bits = np.random.default_rng(0).integers(0, 1 << 23, 1 << 20, dtype=np.uint32)
    edges = np.array([0, 0x7FFF, 0x8000, 0x8001, 0xFFFF, 0x17FFF, 0x18000, 0x7FFFFF, 0x7F8000, 0x7F7FFF], np.uint32)
    x = (np.concatenate([bits, edges]) | np.uint32(0x3F800000)).view(np.float32)  # 1 <= x < 2
    h, m, low = _parts(x)
    assert np.array_equal(_nearest_bf16(low), low)
    assert np.array_equal(h.astype(np.float64) + m + low, x.astype(np.float64))
    assert np.max(np.abs(m)) <= 2.0 ** -8 and np.max(np.abs(low)) <= 2.0 ** -17


def test_products_left_out():
    """m l + l m + l l is at most 2^-24 + 2^-34 of a product, and of either sign."""
    rng = np.random.default_rng(1)
    a, b = ((rng.integers(0, 1 << 23, 1 << 20, dtype=np.uint32) | np.uint32(0x3F800000)).view(np.float32) for _ in "ab")
    (_, ma, la), (_, mb, lb) = ([p.astype(np.float64) for p in _parts(v)] for v in (a, b))
    left = (ma * lb + la * mb + la * lb) / (a.astype(np.float64) * b)
    assert np.max(np.abs(left)) <= 2.0 ** -24 + 2.0 ** -34
    assert abs(left.mean()) <= 5 * left.std() / np.sqrt(left.size)
