"""GPU tests of the grouped linears (cfops_linears_forward / _backward) and the
adapter kernels behind them (cpuforge_amd/csrc/lora.hip, the segmented GEMM of
gemm_f32.hip) against float64: ranks around the 16-wide blocks, token counts
around a chunk, widths around a tile, mixed groups, accumulation and frozen parts."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def close(got, want, terms, mag):
    """f32 sums of `terms` products whose absolute values sum to `mag`, through
    one more such product for an adapter: a rounding per term at most."""
    bound = 2.0 ** -24 * (terms + 16) * mag + 1e-30
    err = (got.double() - want).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


# (t, in, [(out, rank or 0), ...])
CASES = [(1, 5, [(3, 1)]), (63, 31, [(65, 4), (64, 0)]), (64, 576, [(576, 16), (192, 16), (192, 16)]),
         (130, 577, [(33, 17), (130, 33)]), (1000, 96, [(1536, 16), (1536, 16)]), (4096, 64, [(70, 8)]),
         (77, 48, [(64, 3), (64, 16), (64, 20), (64, 0), (40, 5)])]


@pytest.mark.parametrize("acc", [False, True])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"t{c[0]}-in{c[1]}-n{len(c[2])}")
def test_linears_match_f64(case, acc):
    from cpuforge_amd import ops as P
    t, inn, specs = case
    print(t, inn, specs, acc, flush=True)
    g = torch.Generator(device=DEV).manual_seed(t + inn)
    R = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    x, dx0 = R(t, inn), R(t, inn)
    fresh = (lambda z: z.clone()) if acc else (lambda z: torch.full_like(z, float("nan")))
    base = (lambda z: z.double()) if acc else (lambda z: torch.zeros_like(z).double())
    lins, xd = [], x.double()
    for out, r in specs:
        li = dict(w=R(out, inn), scale=0.5, y=torch.full((t, out), float("nan"), device=DEV))
        if r:
            li.update(lora_a=R(r, inn), lora_b=R(out, r), xs=torch.full((t, r), float("nan"), device=DEV))
        lins.append(li)
    P.linears_forward(x, t, inn, lins)
    for li, (out, r) in zip(lins, specs):
        want, mag = xd @ li["w"].double().t(), xd.abs() @ li["w"].double().abs().t()
        if r:
            a, b = li["lora_a"].double(), li["lora_b"].double()
            xs = 0.5 * (xd @ a.t())
            close(li["xs"], xs, inn, 0.5 * (xd.abs() @ a.abs().t()))
            want, mag = want + xs @ b.t(), mag + 0.5 * (xd.abs() @ a.abs().t()) @ b.abs().t()
        close(li["y"], want, 2 * inn + r, mag)
    dx, want, mag, terms = fresh(dx0), base(dx0), base(dx0).abs(), 0
    grads = []
    for i, (li, (out, r)) in enumerate(zip(lins, specs)):
        li["dy"] = R(t, out)
        dyd = li["dy"].double()
        init = dict(gw=R(out, inn))
        want, mag = want + dyd @ li["w"].double(), mag + dyd.abs() @ li["w"].double().abs()
        ref = dict(gw=(base(init["gw"]) + dyd.t() @ xd, base(init["gw"]).abs() + dyd.abs().t() @ xd.abs(), t))
        if r:
            a, b, xs = li["lora_a"].double(), li["lora_b"].double(), li["xs"].double()
            dxa, mdxa = 0.5 * (dyd @ b), 0.5 * (dyd.abs() @ b.abs())
            want, mag = want + dxa @ a, mag + mdxa @ a.abs()
            init.update(ga=R(r, inn), gb=R(out, r))
            ref["ga"] = (base(init["ga"]) + dxa.t() @ xd, base(init["ga"]).abs() + mdxa.t() @ xd.abs(), t + out)
            ref["gb"] = (base(init["gb"]) + dyd.t() @ xs, base(init["gb"]).abs() + dyd.abs().t() @ xs.abs(), t)
        if i % 2:  # frozen base weight, and (rank > 0) a frozen B
            init.pop("gw")
            init.pop("gb", None)
        li.update({n: fresh(z) for n, z in init.items()})
        grads += [(li[n], *ref[n]) for n in init]
        terms += 2 * out + r
    P.linears_backward(x, t, inn, dx, lins, acc=acc)
    # Groups past the fourth linear add to dx once more.
    close(dx, want, terms, mag)
    for got, w, m, n in grads:
        close(got, w, n, m)
    for li in lins:
        for n in ("gw", "ga", "gb"):
            li.pop(n, None)
        if "lora_a" in li:
            li["gb"] = torch.zeros_like(li["lora_b"])
    P.linears_backward(x, t, inn, None, lins)  # no gradient of x, B's only
    for li in lins:
        if "gb" in li:
            dyd, xs = li["dy"].double(), li["xs"].double()
            close(li["gb"], dyd.t() @ xs, t, dyd.abs().t() @ xs.abs())


def test_linears_autograd_unused_output_and_frozen_input():
    """An output that takes no part in the loss leaves zero gradients; an
    input that needs none gets none."""
    from cpuforge_amd import autograd as A
    g = torch.Generator(device=DEV).manual_seed(3)
    R = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    x = R(70, 40).requires_grad_()
    specs = [(R(50, 40), R(8, 40).requires_grad_(), R(50, 8).requires_grad_(), 2.0) for _ in range(2)]
    y0, _ = A.shared_input_linears(x, specs)
    (w, a, b, _), (_, a1, b1, _) = specs
    gx, ga, gb, ga1, gb1 = torch.autograd.grad(y0.sum(), [x, a, b, a1, b1])
    assert not ga1.any() and not gb1.any()
    one = torch.ones(70, 50, dtype=torch.float64, device=DEV)
    assert torch.allclose(gx.double(), one @ w.double() + 2.0 * (one @ b.double()) @ a.double(), rtol=1e-5, atol=1e-4)
    z = A.linear(x.detach(), w, a, b, 2.0)
    ga2, = torch.autograd.grad(z.sum(), [a])
    assert torch.allclose(ga2, ga, rtol=1e-5, atol=1e-4)


def test_linear_functions_by_name():
    """autograd.LinearFn and SharedInputLinearsFn are what linear() and
    shared_input_linears() apply."""
    from cpuforge_amd import autograd as A
    g = torch.Generator(device=DEV).manual_seed(4)
    R = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    x, w, a, b = (t.requires_grad_() for t in (R(2, 9, 40), R(50, 40), R(8, 40), R(50, 8)))
    dy = R(2, 9, 50)
    outs = [A.linear(x, w, a, b, 2.0), A.LinearFn.apply(x, w, a, b, 2.0),
            A.SharedInputLinearsFn.apply(x, (2.0,), w, a, b)[0]]
    grads = [torch.autograd.grad(y, (x, w, a, b), dy) for y in outs]
    for y, got in zip(outs[1:], grads[1:]):
        assert torch.equal(y, outs[0]) and all(torch.equal(p, q) for p, q in zip(got, grads[0]))
    assert A.LinearFn.apply(x, w, None, None, 1.0).shape == (2, 9, 50)


@pytest.mark.parametrize("t,inn,out,r", [((1 << 27) + 50, 2, 1, 1), (3, 2, 2, 65536 * 16 + 3)])
def test_adapter_beyond_one_launch(t, inn, out, r):
    """More tokens, and a higher rank, than the threads and blocks of one launch."""
    from cpuforge_amd import ops as P
    g = torch.Generator(device=DEV).manual_seed(r)
    R = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    x, w, a, b = R(t, inn), R(out, inn), R(r, inn), R(out, r)
    xs, y = torch.full((t, r), float("nan"), device=DEV), torch.full((t, out), float("nan"), device=DEV)
    li = dict(w=w, lora_a=a, lora_b=b, scale=0.5)
    P.linears_forward(x, t, inn, [dict(li, y=y, xs=xs)])
    dy = R(t, out)
    dx, ga, gb = torch.full_like(x, float("nan")), torch.empty_like(a), torch.empty_like(b)
    P.linears_backward(x, t, inn, dx, [dict(li, xs=xs, dy=dy, ga=ga, gb=gb)], acc=False)
    n = min(t, 500)
    for part in (slice(0, n), slice(t - n, t)):
        xd, wxs = x[part].double(), 0.5 * (x[part].double() @ a.double().t())
        close = lambda u, v, m: bool(((u[part] - v).abs() <= 2.0 ** -20 * m + 1e-30).all())  # noqa: E731
        assert close(xs, wxs, xd.abs() @ a.double().abs().t())
        assert close(y, xd @ w.double().t() + wxs @ b.double().t(), 1e3 + wxs.abs() @ b.double().abs().t())
        gd = dy[part].double()
        want = gd @ w.double() + (0.5 * (gd @ b.double())) @ a.double()
        assert close(dx, want, 1e3 + 0.5 * (gd.abs() @ b.double().abs()) @ a.double().abs())
    sums = dy.double().t() @ xs.double()
    assert bool(((gb - sums).abs() <= 1e-4 * sums.abs().max()).all())
    assert bool(ga.isfinite().all())
