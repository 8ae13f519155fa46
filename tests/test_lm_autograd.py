"""The language-model nodes (lm_kernels) under differentiation in earnest: inputs that depend on each
other, tied weights, backwards that are differentiated again.  On the CPU with the HIP passes replaced
by the same in torch operations."""
import pytest
import torch
import torch.nn.functional as F

from conftest import rel_l2


@pytest.fixture
def cpu_passes(monkeypatch):
    """lm_kernels with its HIP passes in torch operations (forward; the backwards under test are those
    that torch differentiates)."""
    from atomic_gdn2 import lm_kernels as K

    def rms(x, scale, gate=None, heads=None):
        if gate is None:
            return K.rms_ref(x, scale)
        B, H, L, D = x.shape
        return K.rms_ref(x.transpose(1, 2).reshape(B * L, H * D), scale) * F.silu(gate)

    def swiglu(gu, d_act=None):
        assert d_act is None
        g, u = gu.chunk(2, dim=1)
        return F.silu(g) * u

    monkeypatch.setattr(K, "_rms", rms)
    monkeypatch.setattr(K, "_swiglu", swiglu)
    monkeypatch.setattr(K, "_gather", lambda parts, ld: F.pad(torch.cat(list(parts), 1), (0, ld - sum(p.shape[1] for p in parts))))
    return K


def _grads(f, leaves, loss=lambda y: y.square().sum()):
    """First-order gradients with create_graph, and those of a scalar of them."""
    first = torch.autograd.grad(loss(f(*leaves)), leaves, create_graph=True)
    second = torch.autograd.grad(sum(g.square().sum() for g in first), leaves, create_graph=True)
    return [t.detach() for t in first + second]


def test_create_graph_with_inputs_that_depend_on_each_other(cpu_passes):
    """_PostMix takes x and two tensors computed from it (the operator's o and the gate's logits): each
    path is counted once.  The same expression in torch operations, float64: 1e-12."""
    K = cpu_passes
    gen = torch.Generator().manual_seed(0)
    r = lambda *s: torch.randn(s, generator=gen, dtype=torch.float64).requires_grad_(True)  # noqa: E731
    B, L, H, D, d = 2, 5, 2, 4, 6
    leaves = [r(B, L, d), r(d, H * D), r(d, H * D), r(H * D), r(H * D, d)]

    def through(node):
        def f(x, wi, wg, scale, wo):
            o = (x @ wi).reshape(B, L, H, D).transpose(1, 2).contiguous()
            return node(o, (x @ wg).reshape(B * L, H * D), x, scale, wo)
        return f

    for a, b in zip(_grads(through(K._PostMix.apply), leaves), _grads(through(K._postmix_ref), leaves)):
        assert rel_l2(a, b) <= 1e-12


def test_create_graph_with_a_tied_weight(cpu_passes):
    """One matrix as both of the MLP's input weights: its two gradients are added once each."""
    K = cpu_passes
    gen = torch.Generator().manual_seed(1)
    r = lambda *s: torch.randn(s, generator=gen, dtype=torch.float64).requires_grad_(True)  # noqa: E731
    leaves = [r(3, 4, 6), r(6), r(6, 8), r(8, 6)]
    tied = lambda node: lambda x, scale, w, wd: node(x, scale, w, w, wd)  # noqa: E731
    for a, b in zip(_grads(tied(K._Mlp.apply), leaves), _grads(tied(K._mlp_ref), leaves)):
        assert rel_l2(a, b) <= 1e-12


@pytest.mark.gpu
def test_block_first_order_gradients_with_create_graph():
    """The whole block: the gradients of a backward that keeps its graph are those of one that does
    not (two float32 evaluations of the same steps, each within about 1e-5 of the exact ones)."""
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")
    from atomic_gdn2 import e2e_lm, lm_kernels
    cfg = e2e_lm.LMConfig(d_model=128, n_heads=3, d_head=64)
    torch.manual_seed(0)
    blk = e2e_lm.GDN2Block(cfg, e2e_lm.blhd_kernel(e2e_lm.operator_cfg(), 64)).cuda()
    x = torch.randn(2, 192, 128, device="cuda", requires_grad=True)
    assert lm_kernels.usable(blk, x, e2e_lm.Dense, e2e_lm.CausalDepthwiseConv, e2e_lm.RMSNorm)
    leaves, w = [x] + list(blk.parameters()), torch.randn(2, 192, 128, device="cuda")
    plain = torch.autograd.grad(blk(x), leaves, w)
    kept = torch.autograd.grad(blk(x), leaves, w, create_graph=True)
    for a, b in zip(kept, plain):
        assert rel_l2(a.detach(), b) <= 2e-5
