"""The native call path (csrc/bind.cpp) against the Python path it stands for: the same bits on plain
calls, and None (so that Python validates, casts and raises) on everything else."""
import types

import pytest
import torch

from test_gpu_parity import base_cfg


def _python_only(monkeypatch):
    from atomic_gdn2 import _lib
    no = types.SimpleNamespace(op=lambda *a: None, sequence=lambda *a: None, decode=lambda *a: None)
    monkeypatch.setattr(_lib, "bind", lambda: no)


def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")


def _xs(shape, dtype=torch.float32, seed=0):
    gen = torch.Generator().manual_seed(seed)
    r = lambda: torch.randn(shape, generator=gen)  # noqa: E731
    xs = [r() * 0.1, r() * 0.1, r(), r(), torch.sigmoid(r()), -0.1 * torch.nn.functional.softplus(r())]
    return [x.to("cuda", dtype) for x in xs]


def _grad(fn, xs, h0, transpose=False):
    xs = [x.detach().clone().requires_grad_(True) for x in xs]
    ins = [x.transpose(1, 2).contiguous().transpose(1, 2) for x in xs] if transpose else xs
    hs = [] if h0 is None else [h0.detach().clone().requires_grad_(True)]
    o, h = fn(*ins, *hs)
    return [o.detach(), h.detach()] + list(torch.autograd.grad((o, h), xs + hs, (o.detach(), h.detach())))


@pytest.mark.gpu
@pytest.mark.parametrize("D,L,kw", [(64, 192, dict(max_chunks_per_call=2)), (128, 256, dict(max_chunks_per_call=1)),
                                    (128, 256, dict(bt=128, bc=64, score_bs=128, wy_eps=1e-3))])
@pytest.mark.parametrize("with_h0", [False, True])
def test_operator_same_bits_as_python(monkeypatch, D, L, kw, with_h0):
    _need_gpu()
    from atomic_gdn2 import make_blr_trainable
    xs = _xs((2, 3, L, D))
    h0 = 0.1 * torch.randn(2, 3, D, D, device="cuda") if with_h0 else None
    run = lambda: (_grad(make_blr_trainable(base_cfg(**kw), 0.1), xs, h0)  # noqa: E731
                   + _grad(make_blr_trainable(base_cfg(**kw), 0.1), xs, h0, transpose=True)
                   + list(make_blr_trainable(base_cfg(**kw), 0.1)(*xs, h0))
                   + list(make_blr_trainable(base_cfg(**kw), 0.1)(*(x.bfloat16() for x in xs), h0)))
    got = run()
    _python_only(monkeypatch)
    want = run()
    for i, (a, b) in enumerate(zip(got, want)):
        assert a.dtype == b.dtype and torch.equal(a, b), i


@pytest.mark.gpu
def test_operator_node_lifetime_hooks_and_partial_gradients():
    """The node outlives the callable that made it, its saved tensors go through saved-tensor hooks,
    only the needed gradients and cotangents take part."""
    _need_gpu()
    from atomic_gdn2 import make_blr_trainable
    xs = _xs((1, 2, 128, 64))
    fn = make_blr_trainable(base_cfg(), 0.1)
    ref = _grad(fn, xs, None)
    seen = []
    ys = [x.clone().requires_grad_(i == 1) for i, x in enumerate(xs)]
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(1), t.clone())[1], lambda t: t):
        o, h = fn(*ys)
    del fn
    assert len(seen) == 7                       # six inputs and the segment's residual
    dk, = torch.autograd.grad((o, h), [ys[1]], (o.detach(), h.detach()))
    assert torch.equal(dk, ref[3])
    z = [x.clone().requires_grad_(True) for x in xs]
    o, h = make_blr_trainable(base_cfg(), 0.1)(*z)
    a = torch.autograd.grad(h, z, h.detach(), retain_graph=True)       # o unused: a zero cotangent
    b = torch.autograd.grad((o, h), z, (torch.zeros_like(o), h.detach()))
    assert all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("fuse,tau", [(False, None), (True, 3.0)])
def test_decode_same_bits_as_python(monkeypatch, dtype, fuse, tau):
    _need_gpu()
    from atomic_gdn2.inference import decode_step
    B, H, D = 5, 3, 64
    xs = _xs((B, H, D), dtype)
    st = (0.3 * torch.randn(B, H, D, D, device="cuda")).to(dtype)
    flags = [0, 1, -3, 7, 0]
    resets = [None, torch.tensor(flags, dtype=torch.int32, device="cuda"),
              torch.tensor(flags, dtype=torch.int64, device="cuda"), torch.tensor(flags, device="cuda") > 0,
              torch.tensor([0, 1, 0, 7, 0], dtype=torch.uint8, device="cuda"),
              torch.tensor(flags, dtype=torch.float32, device="cuda"), flags,
              torch.tensor([[0, 2**32 + 1, -1, 2**31, 2**32]], device="cuda")]
    kw = dict(fuse_prologue=fuse, stability_tau=tau, state_dtype=dtype)
    if fuse:
        kw.update(a_log=torch.linspace(-3, 0, H, device="cuda"), dt_bias=torch.linspace(-1, 1, D, device="cuda"))
    run = lambda: [t for r in resets for t in decode_step(*xs, st, 0.2, reset=r, **kw)]  # noqa: E731
    got = run()
    _python_only(monkeypatch)
    for i, (a, b) in enumerate(zip(got, run())):
        assert a.dtype == b.dtype and torch.equal(a, b), i


@pytest.mark.gpu
def test_refused_calls_reach_python():
    _need_gpu()
    from atomic_gdn2 import make_blr_trainable
    from atomic_gdn2.inference import decode_step
    fn = make_blr_trainable(base_cfg(), 0.1)
    xs = _xs((1, 2, 128, 64))
    with pytest.raises(ValueError, match="divisible"):
        fn(*(x[:, :, :100] for x in xs))
    with pytest.raises(ValueError, match="differs from q.shape"):
        fn(*xs[:5], xs[5][:, :1])
    with pytest.raises(ValueError, match="h0.shape"):
        fn(*xs, torch.zeros(1, 2, 64, 32, device="cuda"))
    with pytest.raises(ValueError, match="empty input"):
        fn(*(x[:0] for x in xs))
    with pytest.raises(ValueError, match="gdn2_fwd"):
        fn(*_xs((1, 1, 64, 96)))
    with pytest.raises(TypeError):
        fn(*(x.long() for x in xs))
    with pytest.raises(ValueError, match="is on"):
        fn(*xs[:5], xs[5].cpu())
    o64, _ = fn(*(x.double() for x in xs))           # other float dtypes are cast
    assert torch.equal(o64, fn(*(x.double().float() for x in xs))[0])
    with pytest.raises(Exception):
        torch.func.vmap(lambda q: fn(q, *xs[1:])[0])(torch.stack([xs[0], xs[0]]))
    with pytest.raises(ValueError, match="state must be"):
        decode_step(*(x[:, :, 0] for x in xs), torch.zeros(1, 2, 64, 32, device="cuda"))
    a = decode_step(*(x[:, :, 3] for x in xs), torch.zeros(1, 2, 64, 64, device="cuda"))     # strided rows are copied
    b = decode_step(*(x[:, :, 3].contiguous() for x in xs), torch.zeros(1, 2, 64, 64, device="cuda"))
    assert all(torch.equal(x, y) for x, y in zip(a, b))


def test_cpu_tensors_are_not_plain():
    from atomic_gdn2 import _lib
    b = _lib.bind()
    op = b.op(bytes(_lib.make_desc(base_cfg(), 0, 0, 0, 0, 0.1, state_ckpt=3)), 2048)
    x = torch.zeros(1, 1, 64, 64)
    assert b.sequence(op, x, x, x, x, x, x, None) is None
    y = torch.zeros(1, 1, 64)
    assert b.decode(y, y, y, y, y, y, x, 1.0, None, False, None, False, None, None) is None
    with pytest.raises(TypeError):
        b.op(b"short", 64)
    with pytest.raises(ValueError):
        b.op(bytes(_lib.make_desc(base_cfg(), 0, 0, 0, 0, 0.1)), 0)
