"""The three-piece bf16 split of f32 values (cpuforge_amd/csrc/split3.hpp) restated
in numpy: what it holds, what its six products leave out, and that the accuracy
checks of the GPU tests fail where a product is missing."""
import numpy as np
import pytest

from test_gpu_f32_split import LSE_LIMIT, O_LIMIT
from test_gpu_gemm import REL_LIMIT

SIX = ((0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0))


def bf16(x):
    """To nearest even, as f32 values."""
    u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7fff + (u >> 16 & 1)) >> 16 << 16).astype(np.uint32).view(np.float32)


def pieces(x, scale=np.float32(65536)):
    r, out = x.astype(np.float32) * scale, []
    for _ in range(3):
        out.append(bf16(r))
        r = r - out[-1]
    return [p.astype(np.float64) / float(scale) for p in out]


def sum_of(products, a, b):
    """Sum over k of the given products of pieces, exact to f64."""
    pa, pb = pieces(a), pieces(b)
    return sum(np.einsum("mk,kn->mn", pa[i], pb[j]) for i, j in products)


def test_pieces_hold_every_bit():
    r = np.random.default_rng(1)
    x = r.standard_normal(200000).astype(np.float32) * np.exp2(r.integers(-149, 108, 200000)).astype(np.float32)
    x = np.concatenate([x, np.float32([0, 1e-45, -1e-45, 1.1754944e-38, 1.0038986, 2.5e33])])
    p = pieces(x)
    assert np.array_equal(p[0] + p[1] + p[2], x.astype(np.float64))
    y = x[np.abs(x) >= 2.0 ** -126].astype(np.float64)
    p = pieces(y)
    assert np.abs(p[1] / y).max() <= 2.0 ** -8 and np.abs(p[2] / y).max() <= 2.0 ** -17
    # Unscaled, values below 2^-110 lose bits.
    small = (r.random(1000) + 1).astype(np.float32) * np.float32(2.0 ** -118)
    assert (sum(pieces(small, np.float32(1))) != small).any() and (sum(pieces(small)) == small).all()


def test_products_left_out():
    """At most about an f32 rounding (2^-24) of |a b|, 2^-28 as a rule."""
    m = (1 + np.arange(2 ** 16) * 2.0 ** -16).astype(np.float32)
    p = pieces(m)
    worst = 2 * np.abs(p[1]) * np.abs(p[2]) + p[2] ** 2
    assert (worst / m.astype(np.float64) ** 2).max() <= 2.0 ** -24
    r = np.random.default_rng(2)
    a, b = (r.standard_normal(100000).astype(np.float32) for _ in range(2))
    pa, pb = pieces(a), pieces(b)
    left = pa[1] * pb[2] + pa[2] * pb[1] + pa[2] * pb[2]
    assert np.sqrt((left ** 2 / (a.astype(np.float64) * b) ** 2).mean()) <= 2.0 ** -26


@pytest.mark.parametrize("k", [576, 4096])
def test_a_missing_product_fails_the_gemm_check(k):
    r = np.random.default_rng(k)
    a, b = r.standard_normal((48, k)).astype(np.float32), r.standard_normal((k, 48)).astype(np.float32)
    want = a.astype(np.float64) @ b.astype(np.float64)
    rel = lambda c: np.linalg.norm(c - want) / np.linalg.norm(want)  # noqa: E731
    assert rel(sum_of(SIX, a, b)) < 0.1 * REL_LIMIT[k]
    for gone in SIX:
        assert rel(sum_of([p for p in SIX if p != gone], a, b)) > 1.5 * REL_LIMIT[k], gone


def test_a_missing_product_fails_the_attention_check():
    r = np.random.default_rng(3)
    S, d = 200, 64
    q, k, v = (r.standard_normal((S, d)).astype(np.float32) for _ in range(3))
    causal = np.tril(np.ones((S, S), bool))

    def attention(qk, pv):
        s = np.where(causal, sum_of(qk, q, k.T) / np.sqrt(d), -np.inf)
        m = s.max(-1, keepdims=True)
        p = np.exp(s - m)
        return sum_of(pv, p.astype(np.float32), v) / p.sum(-1, keepdims=True), (m + np.log(p.sum(-1, keepdims=True)))

    s = np.where(causal, q.astype(np.float64) @ k.T.astype(np.float64) / np.sqrt(d), -np.inf)
    p = np.exp(s)
    want = (p / p.sum(-1, keepdims=True)) @ v.astype(np.float64), np.log(p.sum(-1, keepdims=True))
    rel = lambda x: [np.linalg.norm(a - b) / np.linalg.norm(b) for a, b in zip(x, want)]  # noqa: E731
    o, lse = rel(attention(SIX, SIX))
    assert o < 0.2 * O_LIMIT and lse < 0.2 * LSE_LIMIT
    for gone in SIX:
        fewer = [x for x in SIX if x != gone]
        o, lse = rel(attention(fewer, SIX))
        assert o > 1.5 * O_LIMIT or lse > 1.5 * LSE_LIMIT, ("scores", gone, o, lse)
        assert rel(attention(SIX, fewer))[0] > 1.5 * O_LIMIT, ("values", gone)
