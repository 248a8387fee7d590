"""GPU tests of the overwriting attention backward (cfattn_bwd_grad,
cfattn_fused_bwd_grad): into buffers of NaN it gives what accumulating into
zeros gives, bit for bit up to the sign of a zero, on every kernel that writes
a gradient row (generic, bf16 at both head dims with and without stored dS,
fp32 with one and several key and query splits, the prologue's epilogues and
its own passes), at lengths below, at and beside a tile's edge."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
NAN = float("nan")


def _run(call, sizes):
    """The call's gradients into zeros (accumulating) and into NaN (overwriting)."""
    out = []
    for fill in (0.0, NAN):
        grads = [None if n is None else torch.full((n,), fill, device=DEV) for n in sizes]
        call(fill == 0.0, *[None if g is None else g.data_ptr() for g in grads])
        out.append(grads)
    torch.cuda.synchronize()
    for a, b in zip(*out):
        assert a is None or torch.equal(a, b)


@pytest.mark.parametrize("seq", [1, 31, 128, 333])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("heads,kv,dim", [(6, 2, 6), (4, 4, 80), (9, 3, 64), (32, 8, 64), (8, 2, 128)])
@pytest.mark.parametrize("ds", [True, False])
def test_bwd_grad_equals_accumulating(seq, dtype, heads, kv, dim, ds):
    from cpuforge_amd import _lib
    from cpuforge_amd import device as D
    print(seq, dtype, heads, kv, dim, ds, flush=True)
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    g = torch.Generator(device=DEV).manual_seed(seq * 1000 + heads * 10 + dim)
    R = lambda h: torch.randn(2, seq, h, dim, generator=g, device=DEV).to(dt)  # noqa: E731
    q, k, v, d_o = R(heads), R(kv), R(kv), R(heads)
    ctx = D.Context()
    if not ds:
        _lib.check(ctx._lib.cfattn_set_ds_limit(ctx.handle, 0), ctx.handle)
    o, lse = D.fwd(q, k, v, ctx=ctx)
    B, s = D._batched(q, k)

    def call(acc, *grads):
        fn = ctx._lib.cfattn_bwd if acc else ctx._lib.cfattn_bwd_grad
        _lib.check(fn(ctx.handle, s.c(), B, D._code(q), d_o.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                      o.data_ptr(), lse.data_ptr(), *grads, D._stream()), ctx.handle)

    _run(call, [q.numel(), k.numel(), k.numel()])


@pytest.mark.parametrize("seq", [1, 33, 300])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("heads,kv,dim", [(6, 2, 6), (9, 3, 64), (8, 2, 128), (2, 1, 256)])
@pytest.mark.parametrize("qk_norm", [True, False])
def test_fused_bwd_grad_equals_accumulating(seq, dtype, heads, kv, dim, qk_norm):
    import ctypes

    from cpuforge_amd import RopeCache, _lib
    from cpuforge_amd import device as D
    print(seq, dtype, heads, kv, dim, qk_norm, flush=True)
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    g = torch.Generator(device=DEV).manual_seed(seq * 1000 + heads * 10 + dim)
    R = lambda *sh: torch.randn(*sh, generator=g, device=DEV)  # noqa: E731
    q_pre, k_pre, v, d_o = R(2, seq, heads, dim), R(2, seq, kv, dim), R(2, seq, kv, dim).to(dt), R(2, seq, heads, dim)
    d_o = d_o.to(dt)
    gains = dict(q_norm=1 + 0.1 * R(dim), k_norm=1 + 0.1 * R(dim)) if qk_norm else {}
    pr = D.DeviceRope(RopeCache(dim, seq, 1e4), DEV, **gains)
    ctx = D.Context()
    q, k, q_rstd, k_rstd = D.prologue_fwd(q_pre, k_pre, pr, dtype=dt, ctx=ctx)
    o, lse = D.fwd(q, k, v, ctx=ctx)
    B, s = D._batched(q, k)
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731

    def call(acc, *grads):
        fn = ctx._lib.cfattn_fused_bwd if acc else ctx._lib.cfattn_fused_bwd_grad
        prc = pr.c()
        _lib.check(fn(ctx.handle, s.c(), B, D._code(q), ctypes.byref(prc), d_o.data_ptr(), q_pre.data_ptr(),
                      k_pre.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(),
                      ptr(q_rstd), ptr(k_rstd), *grads, D._stream()), ctx.handle)

    n = dim if qk_norm else None
    _run(call, [q.numel(), k.numel(), k.numel(), n, n])


def test_no_rows_gives_zero_gain_gradients():
    from cpuforge_amd import RopeCache
    from cpuforge_amd import device as D
    pr = D.DeviceRope(RopeCache(64, 4, 1e4), DEV, q_norm=torch.ones(64, device=DEV), k_norm=torch.ones(64, device=DEV))
    e = lambda h: torch.empty(0, 4, h, 64, device=DEV)  # noqa: E731
    rstd = torch.empty(0, device=DEV)
    out = D.fused_bwd(e(4), e(4), e(2), e(4), e(2), e(2), e(4), torch.empty(0, 4, 4, device=DEV), rstd, rstd, pr)
    assert bool((out[3] == 0).all()) and bool((out[4] == 0).all())


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("dim", [6, 64, 128])
@pytest.mark.parametrize("qk_norm", [True, False])
def test_fused_bwd_without_query_heads_adds_nothing(dtype, dim, qk_norm):
    """With n_heads = 0 the accumulating call leaves every gradient as it was
    (and the overwriting one gives zeros), whatever an earlier call left in
    the context's scratch."""
    import ctypes

    from cpuforge_amd import RopeCache, _lib
    from cpuforge_amd import device as D
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    g = torch.Generator(device=DEV).manual_seed(dim)
    R = lambda *sh: torch.randn(*sh, generator=g, device=DEV)  # noqa: E731
    seq, heads, kv = 40, 4, 2
    q_pre, k_pre, v, d_o = R(1, seq, heads, dim), R(1, seq, kv, dim), R(1, seq, kv, dim).to(dt), R(1, seq, heads, dim)
    gains = dict(q_norm=1 + 0.1 * R(dim), k_norm=1 + 0.1 * R(dim)) if qk_norm else {}
    pr = D.DeviceRope(RopeCache(dim, seq, 1e4), DEV, **gains)
    ctx = D.Context()
    o, lse, q, k, q_rstd, k_rstd = D.fused_fwd(q_pre, k_pre, v, pr, ctx=ctx)
    D.fused_bwd(d_o.to(dt), q_pre, k_pre, q, k, v, o, lse, q_rstd, k_rstd, pr, ctx=ctx)  # fills the scratch
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    for acc in (True, False):
        grads = [R(q.numel()), R(k.numel()), R(k.numel())] + ([R(dim), R(dim)] if qk_norm else [None, None])
        before = [None if t is None else t.clone() for t in grads]
        fn = ctx._lib.cfattn_fused_bwd if acc else ctx._lib.cfattn_fused_bwd_grad
        prc = pr.c()
        shape = _lib.Shape(seq, 0, kv, dim)
        _lib.check(fn(ctx.handle, shape, 1, D._code(q), ctypes.byref(prc), d_o.data_ptr(), q_pre.data_ptr(),
                      k_pre.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(),
                      ptr(q_rstd), ptr(k_rstd), *map(ptr, grads), D._stream()), ctx.handle)
        torch.cuda.synchronize()
        assert torch.equal(grads[0], before[0])  # no rows: not touched
        for a, b in zip(grads[1:], before[1:]):
            assert a is None or torch.equal(a, b if acc else torch.zeros_like(b))
