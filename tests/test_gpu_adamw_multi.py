"""GPU test of the batched AdamW (cfops_adamw_update_multi): bit for bit the
per-tensor update, at sizes around its 4096-element blocks and 64-tensor
launches, aligned and not, with frozen and gradientless parameters."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


class Model:
    def __init__(self, named):
        self.named = named

    def named_params(self):
        return iter(self.named)


@pytest.mark.parametrize("count", [1, 63, 64, 65, 200])
def test_batched_adamw_is_bitwise_the_per_tensor_update(count):
    from cpuforge_amd import ops as P
    from cpuforge_amd.optim import AdamW
    g = torch.Generator(device=DEV).manual_seed(count)
    sizes = [1, 3, 4, 4095, 4096, 4097, 8192, 12289, 576, 33]
    named, state, want = [], {}, {}
    for i in range(count):
        n = sizes[i % len(sizes)]
        off = 1 if i % 7 == 3 else 0  # not 16-byte aligned
        p, gr, m, v = (torch.randn(n + off, generator=g, device=DEV)[off:] for _ in range(4))
        v.abs_()
        name = f"layer.{i}." + ("norm" if i % 5 == 0 else "w")
        p.requires_grad_(i % 11 != 10)
        p.grad = None if i % 13 == 12 or not p.requires_grad else gr
        named.append((name, p))
        state[name] = (m, v)
        q, qm, qv = p.detach().clone(), m.clone(), v.clone()
        if p.requires_grad:
            P.adamw_update(q, gr if p.grad is not None else torch.zeros_like(q), qm, qv, 8, 1e-3, 0.9, 0.95, 1e-8,
                           0.0 if "norm" in name else 0.1)
        want[name] = (q, qm, qv)
    opt = AdamW(0.9, 0.95, 1e-8, 0.1)
    opt.step, opt.state = 7, dict(state)
    opt.update(Model(named), 1e-3)
    for name, p in named:
        for a, b in zip((p.detach(), *state[name]), want[name]):
            assert torch.equal(a, b), name


def test_a_tensor_under_two_names_is_updated_twice():
    from cpuforge_amd import ops as P
    from cpuforge_amd.optim import AdamW
    p = torch.ones(100, device=DEV, requires_grad=True)
    p.grad = torch.full((100,), 0.5, device=DEV)
    q = p.detach().clone()
    for _ in range(2):
        z = torch.zeros(100, device=DEV)
        P.adamw_update(q, p.grad, z, torch.zeros(100, device=DEV), 1, 1e-2, 0.9, 0.999, 1e-8, 0.0)
    AdamW(0.9, 0.999, 1e-8, 0.0).update(Model([("a", p), ("b", p)]), 1e-2)
    assert torch.equal(p.detach(), q)


@pytest.mark.parametrize("case", ["view", "inner view", "name", "moments"])
def test_tensors_that_share_memory_are_updated_in_order(case):
    """A parameter beside a view into it, two parameters under one name (and
    so with one state), moments that overlap: as updated one after the other."""
    from cpuforge_amd import ops as P
    from cpuforge_amd.optim import AdamW

    def build():
        g = torch.Generator(device=DEV).manual_seed(5)
        R = lambda n: torch.randn(n, generator=g, device=DEV)  # noqa: E731
        base, n = R(100000), 60000
        cut = {"view": (0, 40000), "inner view": (8, 1000)}.get(case)
        named = [("a", base), ("b", base[cut[0]:cut[1]])] if cut else [("a", base[:n]), ("b", R(n))]
        if case == "name":
            named = [("a", named[0][1]), ("a", named[1][1])]
        named = [("first", R(777))] + named + [("last", R(4097))]
        grads = [R(p.numel()) for _, p in named]
        ms = [R(p.numel()) for _, p in named]
        vs = [R(p.numel()).square() for _, p in named]
        if case == "name":
            ms[2], vs[2] = ms[1], vs[1]
        if case == "moments":
            flat = R(2 * n).square()
            vs[1], vs[2] = flat[:n], flat[4096:4096 + n]
        return named, grads, ms, vs

    named, grads, ms, vs = build()
    for (_, p), g, m, v in zip(named, grads, ms, vs):
        P.adamw_update(p, g, m, v, 3, 1e-2, 0.9, 0.95, 1e-8, 0.1)
    got, grads2, ms2, vs2 = build()
    opt = AdamW(0.9, 0.95, 1e-8, 0.1)
    opt.step = 2
    for i, (name, p) in enumerate(got):
        p = p.detach().requires_grad_()
        p.grad = grads2[i]
        got[i] = (name, p)
        opt.state[name] = (ms2[i], vs2[i])

    class M:
        def named_params(self):
            return iter(got)
    opt.update(M(), 1e-2)
    for (_, p), (_, q), m, m2, v, v2 in zip(named, got, ms, ms2, vs, vs2):
        assert torch.equal(p, q.detach()) and torch.equal(m, m2) and torch.equal(v, v2)
