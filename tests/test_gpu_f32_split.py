"""GPU tests of the fp32 attention forward on split operands
(cpuforge_amd/csrc/attn_f32x3.hpp): accuracy against float64 at the edges of
its 32-key tiles and key splits, and inputs whose bf16 pieces are not finite,
which the f32 unit computes."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def reference(q, k, v):
    """o, lse in float64."""
    B, S, H, d = q.shape
    G = H // k.shape[2]
    q, k, v = (x.double() for x in (q, k, v))
    s = torch.einsum("bshd,bthd->bhst", q, k.repeat_interleave(G, 2)) / math.sqrt(d)
    s.masked_fill_(torch.ones(S, S, device=DEV, dtype=torch.bool).triu(1), -math.inf)
    return (torch.einsum("bhst,bthd->bshd", torch.softmax(s, -1), v.repeat_interleave(G, 2)),
            torch.logsumexp(s, -1))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("shape", [(1, 1, 2, 1), (2, 31, 3, 3), (1, 32, 4, 1), (1, 33, 9, 3), (3, 127, 8, 2),
                                   (1, 129, 4, 4), (2, 300, 6, 2), (1, 1025, 8, 1)])
def test_forward_is_f32_accurate(shape, d):
    from cpuforge_amd import device as D
    B, S, H, K = shape
    print(shape, d, flush=True)
    g = torch.Generator(device=DEV).manual_seed(S + d)
    q, k, v = (torch.randn(B, S, h, d, generator=g, device=DEV) for h in (H, K, K))
    o, lse = D.fwd(q, k, v)
    want, wlse = reference(q, k, v)
    # A score's error is below (d + 8) 2^-24 sum |q k| / sqrt(d) (about d std-1 products), a probability's
    # relative error that and exp2's few ulp; o is a convex mean of v's.
    smax = 4.0 * math.sqrt(d) * (d + 8) * 2.0 ** -24
    assert (o.double() - want).abs().max() <= (2 * smax + 64 * 2.0 ** -24) * v.abs().max()
    assert (lse.double() - wlse).abs().max() <= smax + 2.0 ** -20


# Relative 2-norm error of o and of lse, twice what was measured at S 128 to 1500
# (9.9e-8 to 1.42e-7; 3.7e-8 to 4.6e-8), and the mean relative error of o for
# positive v (measured up to 2.1e-9).
O_LIMIT, LSE_LIMIT, O_BIAS_LIMIT = 2.8e-7, 9.2e-8, 1e-8


@pytest.mark.parametrize("shape", [(128, 9, 3, 64), (129, 16, 8, 128), (512, 9, 3, 64), (700, 4, 4, 128),
                                   (1025, 8, 1, 128), (1500, 8, 2, 64)])
def test_forward_error_is_an_f32_sums(shape):
    """What the bound above is too wide to show: no piece is lost, no sum biased."""
    from cpuforge_amd import device as D
    S, H, K, d = shape
    g = torch.Generator(device=DEV).manual_seed(S)
    q, k, v = (torch.randn(1, S, h, d, generator=g, device=DEV) for h in (H, K, K))
    o, lse = D.fwd(q, k, v)
    want, wlse = reference(q, k, v)
    assert float((o.double() - want).norm() / want.norm()) <= O_LIMIT
    assert float((lse.double() - wlse).norm() / wlse.norm()) <= LSE_LIMIT
    o, _ = D.fwd(q, k, v.abs())
    want, _ = reference(q, k, v.abs())
    assert abs(float(((o.double() - want) / want).mean())) <= O_BIAS_LIMIT


@pytest.mark.parametrize("d", [64, 128])
def test_forward_of_infinite_and_huge_inputs_is_f32s(d):
    """Infinite values give infinities, NaN scores NaN, in the rows that see
    them only.  A large value stays finite up to 2^119: the unnormalised
    probabilities go to 2^8 (the running max moves lazily), so that f32 itself
    overflows on sums past 2^120."""
    from cpuforge_amd import device as D
    S, H = 200, 2
    g = torch.Generator(device=DEV).manual_seed(d)
    q, k, v = (torch.randn(1, S, H, d, generator=g, device=DEV) for _ in range(3))
    base, _ = D.fwd(q, k, v)
    w = v.clone()
    w[0, 40, 0, 3] = 2.0 ** 119
    o, _ = D.fwd(q, k, w)
    want, _ = reference(q, k, w)
    assert torch.isfinite(o).all()
    assert (o.double() - want).abs().max() <= 1e-5 * want.abs().max()
    w[0, 40, 0, 3] = math.inf
    o, _ = D.fwd(q, k, w)
    assert (o[0, 40:, 0, 3] == math.inf).all()
    # (Queries 32..39 share key 40's tile: their masked zero times infinity is
    # NaN in that head dim, in f32 as well.)
    o[0, 32:, 0, 3] = base[0, 32:, 0, 3]
    assert torch.allclose(o, base, rtol=1e-5, atol=1e-5)
    x = k.clone()
    x[0, 70, 1, 5] = math.nan
    o, lse = D.fwd(q, x, v)
    assert torch.isnan(o[0, 70:, 1]).all() and torch.isnan(lse[0, 1, 70:]).all()
    assert torch.allclose(o[0, :70], base[0, :70], rtol=1e-5, atol=1e-5)
    assert torch.allclose(o[0, :, 0], base[0, :, 0], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("exp", [-114, -124, -140])
def test_forward_of_the_smallest_values(d, exp):
    """Inputs down to f32's subnormals keep all their bits: v as o's scale, and
    k beside a q that makes the scores ordinary numbers."""
    from cpuforge_amd import device as D
    g = torch.Generator(device=DEV).manual_seed(d - exp)
    q, k, v = (torch.randn(1, 200, h, d, generator=g, device=DEV) for h in (4, 2, 2))
    w = v * 2.0 ** exp
    o, _ = D.fwd(q, k, w)
    want, _ = reference(q, k, w)
    # Results below f32's smallest normal are rounded to its subnormals, 2^-149 apart.
    assert float((o.double() - want).norm()) <= 5e-7 * float(want.norm()) + 2.0 ** -149 * want.numel() ** 0.5
    kk, qq = k * 2.0 ** max(exp, -124), q * 2.0 ** min(-exp, 124)
    o, lse = D.fwd(qq, kk, v)
    want, wlse = reference(qq, kk, v)
    assert bool(torch.isfinite(o).all())
    assert float((o.double() - want).norm()) <= 5e-7 * float(want.norm())
    assert float((lse.double() - wlse).abs().max()) <= 4e-6


# Relative 2-norm errors (dq, dk, dv) of unit-variance inputs where the forward
# and the backward form the same f32 scores in one chain of sums.
@pytest.mark.parametrize("shape,limits", [((2, 128, 16, 8, 128), (4.42e-7, 4.43e-7, 3.39e-7)),
                                          ((1, 300, 16, 8, 128), (4.79e-7, 4.82e-7, 3.96e-7)),
                                          ((1, 512, 9, 3, 64), (4.28e-7, 4.20e-7, 3.67e-7)),
                                          ((1, 700, 4, 4, 128), (5.22e-7, 5.18e-7, 4.43e-7))])
def test_gradients_no_further_off_than_with_an_f32_forward(shape, limits):
    """The split forward's lse lacks the rounding of the backward's f32 scores;
    what that costs in P is made up for by rounding them less."""
    from cpuforge_amd import device as D
    B, S, H, K, d = shape
    err = torch.zeros(3, dtype=torch.float64)
    for seed in range(3):
        g = torch.Generator(device=DEV).manual_seed(seed)
        q, k, v, d_o = (torch.randn(B, S, h, d, generator=g, device=DEV) for h in (H, K, K, H))
        grads = D.bwd(d_o, q, k, v, *D.fwd(q, k, v))
        leaves = [x.double().requires_grad_() for x in (q, k, v)]
        want = torch.autograd.grad(reference(*leaves)[0], leaves, d_o.double())
        err += torch.tensor([float((a.double() - b).norm() / b.norm()) for a, b in zip(grads, want)]) / 3
    print(shape, err.tolist(), flush=True)
    assert all(e <= m for e, m in zip(err.tolist(), limits))
