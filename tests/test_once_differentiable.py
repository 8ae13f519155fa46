"""A second derivative through the operator raises; a backward that only keeps its graph does not."""
import pytest
import torch

from test_bind import _python_only, _xs
from test_gpu_parity import base_cfg

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("with_h0", [False, True])
def test_operator(monkeypatch, native, with_h0):
    from atomic_gdn2 import make_blr_trainable
    if not native:
        _python_only(monkeypatch)
    fn = make_blr_trainable(base_cfg(max_chunks_per_call=1), 0.1)
    xs = [x.requires_grad_(True) for x in _xs((1, 2, 128, 64))]
    if with_h0:
        xs.append((0.1 * torch.randn(1, 2, 64, 64, device="cuda")).requires_grad_(True))
    loss = lambda: sum(t.square().sum() for t in fn(*xs))  # noqa: E731
    plain = torch.autograd.grad(loss(), xs)
    kept = torch.autograd.grad(loss(), xs, create_graph=True)
    assert all(torch.equal(a, b) for a, b in zip(kept, plain))
    with pytest.raises(RuntimeError, match="once differentiable"):
        torch.autograd.grad(kept[0].sum(), xs[1])
    for form in (lambda t: t, lambda t: t.mT.contiguous().mT):
        kept = torch.autograd.grad(fn(*map(form, xs))[0].sum(), xs, create_graph=True)
        with pytest.raises(RuntimeError, match="once differentiable"):
            kept[2].sum().backward()
    # linear in the cotangents and in nothing else: no derivative either
    kept = torch.autograd.grad(fn(*xs)[0].sum(), xs, create_graph=True)
    with pytest.raises(RuntimeError, match="once differentiable"):
        torch.autograd.grad(kept[2].sum(), xs[0])


def test_block():
    from atomic_gdn2 import e2e_lm
    cfg = e2e_lm.LMConfig(d_model=64, n_heads=1, d_head=64)
    torch.manual_seed(0)
    blk = e2e_lm.GDN2Block(cfg, e2e_lm.blhd_kernel(e2e_lm.operator_cfg(), 64)).cuda()
    x = torch.randn(1, 64, 64, device="cuda", requires_grad=True)
    g, = torch.autograd.grad(blk(x).square().sum(), x, create_graph=True)
    with pytest.raises(RuntimeError, match="once differentiable"):
        torch.autograd.grad(g.square().sum(), x)
    # behind the operator, where no path leads through it, second derivatives are there
    w = blk.down_proj.weight
    g, = torch.autograd.grad(blk(x).square().sum(), w, create_graph=True)
    h, = torch.autograd.grad(g.square().sum(), w)
    assert float(h.norm()) > 0
