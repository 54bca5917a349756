"""The three-part bf16 products of exact mode, emulated in numpy (CPU): the
precision that tests/test_gpu_exact_range.py asks of the kernels is what six of
the nine part products give and is missed without the third parts, and the scale
that the kernels put on their operands keeps every part of every float32 value.
"""
import numpy as np
import pytest

SCALE = np.float32(2.0 ** 16)  # kSplitScale in femtochat_amd/csrc/attn_exact.hpp


def _bf16(x):
    """float32 values rounded to bfloat16 (to nearest even), subnormal ones included."""
    u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
    return ((((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16) & 0xFFFFFFFF).astype(np.uint32).view(np.float32)


def _parts(x):
    h = _bf16(x)
    m = _bf16(x - h)
    return h, m, _bf16(x - h - m)


def _product(a, b, kept):
    """a @ b of float32 arrays from the kept pairs of parts, summed in float64."""
    A, B = _parts(a), _parts(b)
    return sum(A[i].astype(np.float64) @ B[j].astype(np.float64) for i, j in kept).astype(np.float32)


SIX = [(2, 0), (0, 2), (1, 1), (1, 0), (0, 1), (0, 0)]


@pytest.mark.parametrize("kept,low,high", [(SIX, 0.0, 5e-7), ([p for p in SIX if 2 not in p], 3e-6, 1e-4)])
def test_precision(kept, low, high):
    """Errors of O and the gradients of causal attention (2-norm, against
    float64): below a quarter of the kernels' bound of 2e-6 with all six, above
    it without the third parts."""
    T, D = 128, 64
    rng = np.random.Generator(np.random.PCG64(D))
    Q, K, V, dO = (np.clip(rng.standard_normal((T, D), dtype=np.float32), -1.9, 1.9) for _ in range(4))
    hidden = np.triu(np.ones((T, T), bool), 1)

    def attention(product, real):
        S = np.where(hidden, -np.inf, product(Q, K.T.copy()).astype(np.float64) / np.sqrt(D))
        P = np.exp(S - S.max(1, keepdims=True))
        P /= P.sum(1, keepdims=True)
        O = product(P.astype(real), V)
        dP = product(dO, V.T.copy()).astype(np.float64)
        dS = (P * (dP - (dO * O.astype(np.float64)).sum(1, keepdims=True))).astype(real)
        return O, product(dS, K), product(dS.T.copy(), Q), product(P.T.astype(real).copy(), dO)

    exact = attention(lambda a, b: a.astype(np.float64) @ b.astype(np.float64), np.float64)
    for x, y in zip(attention(lambda a, b: _product(a, b, kept), np.float32), exact):
        assert low <= np.linalg.norm(x - y) / np.linalg.norm(y) <= high


def test_scaled_values_are_the_sum_of_their_parts():
    """Exactly, over all of float32 below 2^111, subnormal values included."""
    rng = np.random.Generator(np.random.PCG64(1))
    bits = rng.integers(0, 1 << 31, 1 << 20, dtype=np.uint32)
    x = np.concatenate([bits, np.arange(1, 1 << 16, dtype=np.uint32), np.uint32(1 << 23) - np.arange(1, 1 << 16, dtype=np.uint32)])
    x = x.view(np.float32)
    x = x[np.isfinite(x) & (x < 2.0 ** 111)]
    h, m, l = _parts(x * SCALE)
    total = h.astype(np.float64) + m + l
    assert np.array_equal(total, x.astype(np.float64) * float(SCALE))
    assert not np.array_equal(sum(p.astype(np.float64) for p in _parts(x)), x.astype(np.float64))  # without the scale
