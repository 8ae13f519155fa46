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


def _hooks(pack):
    return torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t)


@pytest.mark.parametrize("pack", [lambda t: t.to(torch.bfloat16), lambda t: t.flip(0).flip(0).mT.contiguous().mT if t.dim() > 1 else t])
def test_saved_tensors_in_another_form_reach_the_kernels_dense(cpu_passes, monkeypatch, pack):
    """What saved-tensor hooks give back need not be what was saved: the backward kernels, which take
    addresses, get dense float32 tensors of the saved shapes."""
    K = cpu_passes
    seen = []

    def checked(*ts):
        for t in ts:
            assert t is None or (t.dtype == torch.float32 and t.is_contiguous())
            seen.append(t)

    def rms_bwd(x, scale, dy, gate=None, heads=None, res=None):
        checked(x, scale, dy, gate, res)
        return torch.zeros_like(x), torch.zeros_like(scale), None if gate is None else torch.zeros_like(gate)

    def swiglu(gu, d_act=None):
        checked(gu, d_act)
        g, u = gu.chunk(2, dim=1)
        return F.silu(g) * u if d_act is None else torch.zeros_like(gu)

    monkeypatch.setattr(K, "_rms_bwd", rms_bwd)
    monkeypatch.setattr(K, "_swiglu", swiglu)
    monkeypatch.setattr(K, "_scatter", lambda wide, like: [torch.zeros_like(t) for t in like])
    r = lambda *s: torch.randn(s).requires_grad_(True)  # noqa: E731
    for node, xs in [(K._PostMix, [r(2, 2, 5, 4), r(10, 8), r(2, 5, 6), r(8), r(8, 6)]),
                     (K._Mlp, [r(2, 5, 6), r(6), r(6, 8), r(6, 8), r(8, 6)]), (K._RmsNorm, [r(2, 5, 6), r(6)])]:
        with _hooks(pack):
            y = node.apply(*xs)
        seen.clear()
        torch.autograd.grad(y, xs, torch.ones_like(y))
        assert len(seen) >= 3


def test_saved_tensors_of_another_shape_are_refused(cpu_passes):
    K = cpu_passes
    xs = [torch.randn(2, 5, 6, requires_grad=True), torch.randn(6, requires_grad=True)]
    with _hooks(lambda t: t[:1]):
        y = K._RmsNorm.apply(*xs)
    with pytest.raises(RuntimeError, match="saved-tensor hooks"):
        torch.autograd.grad(y, xs, torch.ones_like(y))


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
def test_operator_with_saved_tensors_in_another_form(monkeypatch, native):
    """The operator's node: inputs given back in bfloat16 (here bfloat16 values, so nothing is lost) are
    widened, and a residual of another size is refused."""
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")
    from atomic_gdn2 import make_blr_trainable
    from test_bind import _python_only, _xs
    from test_gpu_parity import base_cfg
    if not native:
        _python_only(monkeypatch)
    fn = make_blr_trainable(base_cfg(max_chunks_per_call=1), 0.1)
    xs = [x.bfloat16().float().requires_grad_(True) for x in _xs((1, 2, 128, 64))]

    def grads(pack):
        with _hooks(pack):
            o, h = fn(*xs)
        return torch.autograd.grad((o, h), xs, (o.detach(), h.detach()))

    want = grads(lambda t: t)
    for pack in (lambda t: t.bfloat16() if t.is_floating_point() else t,
                 lambda t: t.mT.contiguous().mT if t.is_floating_point() else t):
        assert all(torch.equal(a, b) for a, b in zip(grads(pack), want))
    for pack in (lambda t: t if t.is_floating_point() else t[:-256], lambda t: t[:, :1] if t.is_floating_point() else t):
        with pytest.raises(RuntimeError, match="saved-tensor hooks"):
            grads(pack)
