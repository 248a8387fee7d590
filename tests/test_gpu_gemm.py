"""GPU tests of the f32 GEMM kernels (cpuforge_amd/csrc/gemm_f32.hip) at the
edges of their tiles (64, 128, 256), steps (32 k) and splits, against float64,
and on inputs whose bf16 pieces are not finite."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def product(kind, a, b, c, acc):
    from cpuforge_amd import ops as P
    m, n, k = c.shape[0], c.shape[1], a.shape[1]
    if kind == "nn":
        P.matmul_nn(a.contiguous(), b.contiguous(), c, m, k, n, acc)
    elif kind == "nt":
        P.matmul_nt(a.contiguous(), b.t().contiguous(), c, m, k, n, acc)
    else:
        P.matmul_tn(a.t().contiguous(), b.contiguous(), c, m, k, n, acc)
    return c


def check(kind, m, k, n, acc=False, scale_a=1.0, seed=1):
    g = torch.Generator(device=DEV).manual_seed(seed)
    a = torch.randn(m, k, generator=g, device=DEV) * scale_a
    b = torch.randn(k, n, generator=g, device=DEV)
    c0 = torch.randn(m, n, generator=g, device=DEV)
    c = product(kind, a, b, c0.clone() if acc else torch.full((m, n), float("nan"), device=DEV), acc)
    want = a.double() @ b.double() + (c0.double() if acc else 0)
    # Sums in f32: at most one rounding of the partial sum per term (six per 16
    # in one instruction chain, plus the splits' sums and the last one), each
    # 2^-24 of it; the products left out are at most 2^-24 of |a b|.
    bound = 2.0 ** -24 * (k + 8) * (a.abs().double() @ b.abs().double()) + 2.0 ** -22 * want.abs()
    err = (c.double() - want).abs()
    assert bool((err <= bound).all()), (kind, m, k, n, float((err / bound).max()))


@pytest.mark.parametrize("kind", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (63, 7, 65), (64, 8, 64), (65, 31, 63), (127, 32, 129), (129, 33, 127),
                                   (257, 100, 130), (255, 64, 383), (1, 1537, 300), (70, 4099, 5), (300, 1333, 501),
                                   (4096, 96, 576), (4100, 160, 700), (2048, 1000, 2050)])
def test_gemm_edges_match_f64(kind, m, k, n):
    print(kind, m, k, n, flush=True)
    check(kind, m, k, n)
    check(kind, m, k, n, acc=True)


# Relative 2-norm error of normal values by k, twice what was measured (7.8e-8 to
# 1.36e-7 at k = 576, 1.2e-7 to 2.2e-7 at k = 4096, 2.7e-7 at 49152), and the mean
# relative error of positive ones (measured up to 1.2e-9; 4e-8 and more where
# the leading product shares its sums with the other five).
REL_LIMIT = {576: 2.8e-7, 4096: 4.4e-7, 49152: 5.4e-7}
BIAS_LIMIT = 1e-8


@pytest.mark.parametrize("kind", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,k,n", [(64, 576, 64), (300, 576, 500), (4096, 576, 1536), (64, 4096, 64),
                                   (2048, 4096, 1030), (128, 49152, 576)])
def test_gemm_error_is_an_f32_sums(kind, m, k, n):
    """What the bounds above are too wide to show, on every tile and with the
    contraction split: no piece is lost, and no sum is biased."""
    g = torch.Generator(device=DEV).manual_seed(m + k)
    a, b = torch.randn(m, k, generator=g, device=DEV), torch.randn(k, n, generator=g, device=DEV)
    c, want = product(kind, a, b, torch.empty(m, n, device=DEV), False).double(), a.double() @ b.double()
    assert float((c - want).norm() / want.norm()) <= REL_LIMIT[k]
    a, b = a.abs(), b.abs()
    c, want = product(kind, a, b, torch.empty(m, n, device=DEV), False).double(), a.double() @ b.double()
    assert abs(float(((c - want) / want).mean())) <= BIAS_LIMIT


def test_gemm_rows_longer_than_32_bit_offsets():
    """A row stride of more than 2^22 values: 256 rows of it pass 2^32 bytes."""
    check("nt", 65, (1 << 22) + 5, 3)


def test_gemm_few_rows_of_long_strides():
    """B rows more than 2^26 values apart: 12 of them pass 2^32 bytes."""
    from cpuforge_amd import ops as P
    m, k, n = 3, 21, (1 << 26) + 3
    g = torch.Generator(device=DEV).manual_seed(2)
    a, b = torch.randn(m, k, generator=g, device=DEV), torch.randn(k, n, generator=g, device=DEV)
    c = torch.full((m, n), float("nan"), device=DEV)
    P.matmul_nn(a, b, c, m, k, n, False)
    for part in (slice(0, 1000), slice(n - 1000, n)):
        ad, bd = a.double(), b[:, part].double()
        assert bool(((c[:, part] - ad @ bd).abs() <= 2.0 ** -24 * (k + 8) * (ad.abs() @ bd.abs())).all())


@pytest.mark.parametrize("kind", ["nn", "nt"])
@pytest.mark.parametrize("m", [1, 15, 16, 17, 40])
@pytest.mark.parametrize("k,n", [(16, 16), (15, 17), (512, 33), (513, 15), (531, 700), (1100, 48)])
def test_gemm_few_rows(kind, m, k, n):
    """The kernel for few rows at the edges of its 16 x 16 tiles, its runs of 16
    k and its batches of 512."""
    print(kind, m, k, n, flush=True)
    check(kind, m, k, n)
    check(kind, m, k, n, acc=True)


@pytest.mark.parametrize("kind", ["nn", "nt", "tn"])
def test_gemm_small_and_large_magnitudes(kind):
    """Inputs whose low pieces are bf16 subnormals keep their products'
    accuracy; inputs near the f32 maximum round to infinity in bf16 and take
    the f32 recomputation."""
    check(kind, 70, 96, 66, scale_a=2.0 ** -108)
    g = torch.Generator(device=DEV).manual_seed(3)
    a = torch.randn(70, 96, generator=g, device=DEV)
    b = torch.randn(96, 66, generator=g, device=DEV) * 2.0 ** -20
    a[5, 7] = 3.4028e38  # rounds to infinity in bf16
    c = product(kind, a, b, torch.empty(70, 66, device=DEV), False)
    want = a.double() @ b.double()
    assert bool(torch.isfinite(c).all())
    bound = 2.0 ** -24 * 104 * (a.abs().double() @ b.abs().double())
    assert bool(((c.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("kind", ["nn", "nt", "tn"])
@pytest.mark.parametrize("exp", [-112, -118, -124, -130, -140])
def test_gemm_of_the_smallest_values(kind, exp):
    """Inputs down to f32's subnormals keep all their bits (their low pieces
    would lie below bf16's smallest subnormal): against large ones on the other
    side, the products are ordinary numbers."""
    g = torch.Generator(device=DEV).manual_seed(-exp)
    a = torch.randn(70, 96, generator=g, device=DEV) * 2.0 ** exp
    b = torch.randn(96, 66, generator=g, device=DEV) * 2.0 ** 90
    assert bool((a[:, :8] != 0).any())
    for x, y in ((a, b), (b.t().contiguous(), a.t().contiguous())):
        c = product(kind, x, y, torch.empty(x.shape[0], y.shape[1], device=DEV), False)
        bound = 2.0 ** -24 * 104 * (x.abs().double() @ y.abs().double())
        assert bool(((c.double() - x.double() @ y.double()).abs() <= bound).all())


@pytest.mark.parametrize("kind", ["nn", "nt", "tn"])
def test_gemm_infinities_and_nan_are_f32s(kind):
    """What f32 arithmetic gives where an input is infinite or NaN: the same
    infinities and NaN, the other outputs untouched by them."""
    a = np.ones((70, 40), np.float32)
    b = np.ones((40, 66), np.float32)
    a[3, 2], a[9, 39], a[65, 0] = np.inf, np.nan, -np.inf
    b[5, 1], b[2, 4] = np.inf, 0.0
    with np.errstate(invalid="ignore"):
        want = a @ b
    c = product(kind, torch.from_numpy(a).to(DEV), torch.from_numpy(b).to(DEV), torch.empty(70, 66, device=DEV), False)
    got = c.cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.array_equal(got[ok], want[ok])


@pytest.mark.parametrize("kind", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,k,n", [(70, 37, 66), (65, 4099, 63), (300, 1333, 501), (2048, 1000, 2050), (4096, 96, 2050)])
def test_gemm_recomputed_tiles(kind, m, k, n):
    """Every tile and split form with NaN, infinite and huge values in some
    places: what f32 arithmetic gives there, and its accuracy everywhere else."""
    g = torch.Generator(device=DEV).manual_seed(m + k + n)
    a = torch.randn(m, k, generator=g, device=DEV)
    b = torch.randn(k, n, generator=g, device=DEV)
    a[m - 1, k // 2], a[m // 2, k - 1], a[3, 0], b[k - 1, n - 1] = float("nan"), float("inf"), 2.0 ** 120, -float("inf")
    want = a.double() @ b.double()
    c = product(kind, a, b, torch.empty(m, n, device=DEV), False)
    assert torch.equal(c.isnan(), want.isnan())
    assert torch.equal(c == float("inf"), want == float("inf"))
    assert torch.equal(c == -float("inf"), want == -float("inf"))
    ok = want.isfinite()
    fin = lambda x: torch.where(x.isfinite(), x, 0.0).abs().double()  # noqa: E731
    bound = 2.0 ** -24 * (k + 8) * (fin(a) @ fin(b)) + 2.0 ** -22 * want.abs()
    assert bool(((c.double() - want).abs() <= bound)[ok].all())
