"""GPU test of the cross-entropy row kernel at the edges of its forms (8, 12 or
16 float4 a thread, 512 or 1024 threads, and the streamed one), in place and
not, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("vocab", [4, 2048, 16384, 16388, 32768, 32772, 49148, 49152, 49156, 65536, 65540, 16385])
def test_cross_entropy_rows_at_form_edges(vocab):
    from cpuforge_amd import ops as P
    print(vocab, flush=True)
    g = torch.Generator(device=DEV).manual_seed(vocab)
    rows = 7
    x = torch.randn(rows, vocab, generator=g, device=DEV) * 2
    t = torch.tensor([0, vocab - 1, -100, vocab // 2, min(vocab - 1, 4095), max(0, vocab - 5), 1], device=DEV)
    n = rows - 1
    p = torch.softmax(x.double(), -1)
    want = p / n
    scored = t != -100
    want[scored, t[scored]] -= 1.0 / n
    want[~scored] = 0.0
    loss_want = -torch.log_softmax(x.double(), -1)[scored, t[scored]].mean()
    out = torch.full_like(x, float("nan"))
    loss = P.cross_entropy_fwd_bwd(x, t, out, rows, vocab)
    # expf of the difference (its rounding, at most 2^-24 of 32, and two ulp), a
    # tree sum of about 12 + 10 + 4 levels or, streamed, vocab / 512 in a row, and
    # four more roundings; the target's difference rounds at 1 / n.
    rel = (32 + 2 + 26 + vocab / 512 + 4) * 2.0 ** -24
    bound = rel * p / n
    bound[scored, t[scored]] += 2.0 ** -23 / n
    assert bool(((out.double() - want).abs() <= bound + 1e-37).all())
    assert abs(loss - float(loss_want)) <= (rel + 2.0 ** -22) * (1 + abs(float(loss_want)))
    loss2 = P.cross_entropy_fwd_bwd(x, t, x, rows, vocab)
    assert loss2 == loss and torch.equal(x, out)
