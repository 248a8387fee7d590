"""GPU tests of the overwriting gradients (rmsnorm_backward, silu_mul_backward
with acc=False) and of the one-wave-per-row RMSNorm backward at the edges of
its widths (256 floats to a register step) and row blocks (8), against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rows", [1, 7, 8, 9, 1000])
@pytest.mark.parametrize("dim", [4, 252, 256, 260, 512, 576, 768, 772, 1024, 1028, 2048, 2052, 577])
def test_rmsnorm_backward_edges(rows, dim):
    from cpuforge_amd import ops as P
    print(rows, dim, flush=True)
    g = torch.Generator(device=DEV).manual_seed(rows * 10000 + dim)
    R = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    dy, x, w, dx0, dw0 = R(rows, dim), R(rows, dim), R(dim), R(rows, dim), R(dim)
    y, rstd = torch.empty_like(x), torch.empty(rows, device=DEV)
    P.rmsnorm_forward(x, w, y, rstd, rows, dim, 1e-5)
    xd, wd, dyd, inv = x.double(), w.double(), dy.double(), rstd.double()[:, None]
    xh = xd * inv
    gx = inv * (dyd * wd - xh * (dyd * wd * xh).mean(-1, keepdim=True))
    gw = (dyd * xh).sum(0)
    mag = inv * ((dyd * wd).abs() + xh.abs() * (dyd * wd * xh).abs().mean(-1, keepdim=True))
    wmag = (dyd * xh).abs().sum(0)
    for acc in (True, False):
        for frozen in (True, False):
            dx = dx0.clone() if acc else torch.full_like(x, float("nan"))
            dw = None if frozen else dw0.clone() if acc else torch.full_like(w, float("nan"))
            P.rmsnorm_backward(dy, x, w, rstd, dx, dw, rows, dim, acc=acc)
            # A rounding per term of each sum, and a few per element.
            base = dx0.double() if acc else 0.0
            assert bool(((dx - (gx + base)).abs() <= 2.0 ** -24 * ((dim + 16) * mag + 2 * dx0.abs())).all())
            if not frozen:
                base = dw0.double() if acc else 0.0
                assert bool(((dw - (gw + base)).abs() <= 2.0 ** -24 * ((rows + 16) * wmag + 2 * dw0.abs())).all())


@pytest.mark.parametrize("n", [1, 4, 1001, 4096])
def test_silu_mul_backward_overwrites(n):
    from cpuforge_amd import ops as P
    g = torch.Generator(device=DEV).manual_seed(n)
    dh, a, u = (torch.randn(n, generator=g, device=DEV) for _ in range(3))
    zeros = [torch.zeros(n, device=DEV) for _ in range(2)]
    P.silu_mul_backward(dh, a, u, *zeros)
    out = [torch.full((n,), float("nan"), device=DEV) for _ in range(2)]
    P.silu_mul_backward(dh, a, u, *out, acc=False)
    assert all(torch.equal(x, z) for x, z in zip(out, zeros))


def test_gradients_of_no_rows_are_zero():
    """A sum over no rows overwrites its gradient with zeros, as a zeroed buffer left it."""
    from cpuforge_amd import autograd as A
    from cpuforge_amd import ops as P
    nan = lambda *s: torch.full(s, float("nan"), device=DEV)  # noqa: E731
    x = torch.empty(0, 24, device=DEV)
    dw = nan(24)
    P.rmsnorm_backward(x, x, torch.ones(24, device=DEV), torch.empty(0, device=DEV), torch.empty_like(x), dw, 0, 24,
                       acc=False)
    assert bool((dw == 0).all())
    w, a, b = (torch.randn(*s, device=DEV) for s in ((40, 24), (4, 24), (40, 4)))
    li = dict(w=w, lora_a=a, lora_b=b, scale=2.0, xs=torch.empty(0, 4, device=DEV), dy=torch.empty(0, 40, device=DEV),
              gw=nan(40, 24), ga=nan(4, 24), gb=nan(40, 4))
    P.linears_backward(x, 0, 24, torch.empty_like(x), [li], acc=False)
    assert all(bool((li[n] == 0).all()) for n in ("gw", "ga", "gb"))
    leaves = [t.requires_grad_() for t in (w, a, b)]
    grads = torch.autograd.grad(A.linear(x, w, a, b, 2.0).sum(), leaves)
    assert all(bool((g == 0).all()) for g in grads)
    dx = nan(5, 24)
    P.linears_backward(torch.randn(5, 24, device=DEV), 5, 24, dx, [], acc=False)  # of no linears
    assert bool((dx == 0).all())


def test_rmsnorm_backward_of_more_rows_than_a_launch_has_waves():
    """2^27 rows and more: one wave to two rows would be 2^32 threads."""
    from cpuforge_amd import ops as P
    rows, dim = (1 << 27) + 100, 4
    g = torch.Generator(device=DEV).manual_seed(1)
    x, dy = (torch.randn(rows, dim, generator=g, device=DEV) for _ in range(2))
    w = torch.tensor([1.0, 0.5, -2.0, 1.5], device=DEV)
    rstd, dx = torch.empty(rows, device=DEV), torch.full_like(x, float("nan"))
    y = torch.empty_like(x)
    P.rmsnorm_forward(x, w, y, rstd, rows, dim, 1e-5)
    P.rmsnorm_backward(dy, x, w, rstd, dx, None, rows, dim, acc=False)
    for part in (slice(0, 1000), slice(rows - 1000, rows)):
        xd, gd, inv = x[part].double(), dy[part].double(), rstd[part].double()[:, None]
        xh = xd * inv
        want = inv * (gd * w.double() - xh * (gd * w.double() * xh).mean(-1, keepdim=True))
        mag = inv * ((gd * w).abs() + xh.abs() * (gd * w * xh).abs().mean(-1, keepdim=True))
        assert bool(((dx[part] - want).abs() <= 2.0 ** -24 * 20 * mag).all())
    assert not bool(dx.isnan().any())
