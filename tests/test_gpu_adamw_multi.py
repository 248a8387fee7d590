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
