"""FP32 products on three bf16 parts, emulated on the CPU: the bounds that the
GPU tests hold the kernels to tell a lost product from rounding.

split_operand and split_product (csrc/device_common.hpp): a value is three
parts, each the bf16 rounding of what the ones before it left, and a product
is the sum of six of the nine products of parts.
"""

import numpy as np
import pytest

# rms error of a sum over rms of sum |x w|: at most K roundings, each by up to
# 2^-24 of a partial sum, and those of K terms of random sign are about
# 1.5 / sqrt(K) of sum |x w|
ROUNDING = 1.5 * 2.0 ** -24

SIX = [(0, 2), (2, 0), (1, 1), (0, 1), (1, 0), (0, 0)]


def _bf16(x):
    u = np.ascontiguousarray(x, np.float32).view(np.uint32)
    return ((u + 0x7fff + ((u >> 16) & 1)) & np.uint32(0xffff0000)).view(np.float32)


def _split(x):
    a = _bf16(x)
    b = _bf16(x - a)
    return [p.astype(np.float64) for p in (a, b, x - a - b)]


def _operands(K, seed=0):
    rng = np.random.default_rng(seed)
    return rng.normal(size=(300, K)).astype(np.float32), (rng.normal(size=(K, 128)) / np.sqrt(K)).astype(np.float32)


def _linear(x, w, products):
    X, W = _split(x), _split(w)
    y = np.zeros((len(x), w.shape[1]), np.float32)
    for c in range(0, x.shape[1], 32):  # an MFMA's 32 inputs, its accumulator rounded to FP32
        for i, j in products:
            y = (y + X[i][:, c:c + 32] @ W[j][c:c + 32]).astype(np.float32)
    return y


def test_three_parts_are_exact():
    x, _ = _operands(256)
    parts = _split(x)
    assert np.array_equal(sum(parts), x.astype(np.float64))
    assert all(np.array_equal(_bf16(p.astype(np.float32)), p) for p in parts)
    # the products left out reach 2^-24 of a product, and no more
    one = np.float32(1.0038986)
    p = _split(np.full(1, one))
    assert 2.0 ** -24.1 < abs(float((p[1] * p[2] * 2 + p[2] * p[2])[0])) / float(one) ** 2 < 2.0 ** -24


@pytest.mark.parametrize("K", [32, 40, 128, 256, 768])
def test_a_lost_product_exceeds_the_rounding_bound(K):
    x, w = _operands(K)
    ref = x.astype(np.float64) @ w.astype(np.float64)
    scale = np.sqrt(np.mean((np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64)) ** 2))

    def error(products):
        return np.sqrt(np.mean((_linear(x, w, products) - ref) ** 2)) / scale

    assert error(SIX) < ROUNDING / 4
    for lost in SIX:
        assert error([p for p in SIX if p != lost]) > 1.5 * ROUNDING
