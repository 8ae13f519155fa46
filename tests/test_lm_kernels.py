"""The language-model block's HIP passes (lm_kernels) against the same block in torch operations, and
where the module forward has to stay in charge."""
import dataclasses
import functools

import pytest
import torch

from conftest import rel_l2


def _block(cfg, op, seed=0):
    from atomic_gdn2 import e2e_lm
    torch.manual_seed(seed)
    blk = e2e_lm.GDN2Block(cfg, op)
    with torch.no_grad():                     # biases and scales off their initial constants
        for n, p in blk.named_parameters():
            if p.dim() == 1:
                p.add_(0.1 * torch.randn_like(p))
    return blk


def _passes(cfg, B, L, dev, dtype):
    """The three nodes' references and inputs, without the operator between them."""
    from atomic_gdn2 import lm_kernels as K
    blk = _block(cfg, None).to(dtype)
    gen = torch.Generator().manual_seed(3)
    r = lambda *s: torch.randn(s, generator=gen).to(dtype)  # noqa: E731
    H, D, C = cfg.n_heads, cfg.d_head, cfg.proj_dim
    m = blk
    pre = [2.0 * r(B, L, cfg.d_model)] + [p.detach() for p in (
        m.q_proj.weight, m.k_proj.weight, m.v_proj.weight, m.erase_gate.weight, m.write_gate.weight, m.out_gate.weight,
        m.decay_proj.weight, m.q_conv.weight, m.q_conv.bias, m.k_conv.weight, m.k_conv.bias, m.v_conv.weight,
        m.v_conv.bias, m.erase_gate.bias, m.write_gate.bias, m.decay_proj.bias, m.decay_a)]
    post = [r(B, H, L, D), r(B * L, C), r(B, L, cfg.d_model), m.mixer_out_norm.scale.detach(), m.out_proj.weight.detach()]
    mlp = [r(B, L, cfg.d_model)] + [p.detach() for p in (m.mlp_norm.scale, m.gate_proj.weight, m.up_proj.weight,
                                                         m.down_proj.weight)]
    steps = [(K._premix_ref(H, D, cfg.g_max), lambda *a: K._PreMix.apply(H, D, cfg.g_max, *a), pre),
             (K._postmix_ref, K._PostMix.apply, post), (K._mlp_ref, K._Mlp.apply, mlp),
             (K.rms_ref, K._RmsNorm.apply, [mlp[0], mlp[1]])]
    return [(ref, fused, [t.to(dev).clone().requires_grad_(True) for t in xs]) for ref, fused, xs in steps]


def _run(fn, xs, seed):
    outs = fn(*xs)
    outs = outs if isinstance(outs, tuple) else (outs,)
    gen = torch.Generator().manual_seed(seed)
    ws = [torch.randn(o.shape, generator=gen, dtype=torch.float64).to(o.device, o.dtype) for o in outs]
    return [o.detach() for o in outs] + list(torch.autograd.grad(outs, xs, ws))


def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")


# token counts around the 128-token tile and the runs of 16 / 8 tokens inside it; C and d_model at
# and off whole 256-float wave rows; both head sizes
@pytest.mark.gpu
@pytest.mark.parametrize("B,L,H,D,d", [(1, 5, 1, 64, 4), (2, 3, 1, 128, 64), (1, 127, 3, 64, 260), (3, 130, 6, 128, 512),
                                       (2, 128, 5, 64, 96), (1, 271, 8, 128, 1024)])
def test_passes_match_float64(B, L, H, D, d):
    """float32 chains of a few dozen operations and sums of up to 1024 x 400 terms in blocks: 1e-5 of
    the float64 result."""
    _need_gpu()
    from atomic_gdn2 import e2e_lm
    cfg = e2e_lm.LMConfig(d_model=d, n_heads=H, d_head=D)
    # the same float32 inputs on both sides
    for (ref, _, xs), (_, fused, ys) in zip(_passes(cfg, B, L, "cpu", torch.float32), _passes(cfg, B, L, "cuda", torch.float32)):
        w = _run(ref, [x.detach().double().requires_grad_(True) for x in xs], 5)
        got = _run(fused, ys, 5)
        assert len(got) == len(w)
        for i, (a, b) in enumerate(zip(got, w)):
            assert a.shape == b.shape
            assert rel_l2(a, b) <= 1e-5, (i, rel_l2(a, b))


@pytest.mark.gpu
def test_saturated_and_non_finite_rows():
    """Logits beyond the exponentials' range, infinities and NaN: finite and non-finite entries where
    torch's operations have them, the finite ones within 1e-5."""
    _need_gpu()
    from atomic_gdn2 import e2e_lm
    from atomic_gdn2 import lm_kernels as K
    gen = torch.Generator(device="cuda").manual_seed(0)
    gu = torch.randn(64, 512, generator=gen, device="cuda")
    for j, v in enumerate((120.0, -120.0, 1e4, -1e4, float("inf"), float("-inf"), float("nan"), 0.0)):
        gu[j, 5] = v
        gu[j, 300] = v
    g, u = gu[:, :256], gu[:, 256:]
    want, got = torch.nn.functional.silu(g) * u, K._swiglu(gu)
    assert torch.equal(torch.isnan(want), torch.isnan(got)) and torch.equal(torch.isinf(want), torch.isinf(got))
    ok = torch.isfinite(want)
    assert float((want[ok] - got[ok]).norm() / want[ok].norm()) <= 1e-6
    cfg = e2e_lm.LMConfig(d_model=64, n_heads=2, d_head=64)
    (ref, fused, xs), = _passes(cfg, 1, 40, "cuda", torch.float32)[:1]
    with torch.no_grad():
        xs[0][0, 7] = 1e4
        xs[0][0, 20] = float("nan")
    for a, b in zip(*([t.detach() for t in f(*xs)] for f in (fused, ref))):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isinf(a), torch.isinf(b))
        ok = torch.isfinite(b)
        assert float((a[ok] - b[ok]).norm()) <= 1e-5 * float(b[ok].norm()) + 1e-30


@pytest.mark.gpu
def test_block_is_the_module_forward():
    """The whole block through the HIP passes against the module's own forward (same operator), values
    and all gradients; and the RMS norm's backward that is differentiated again (the other nodes':
    test_lm_autograd.py)."""
    _need_gpu()
    from atomic_gdn2 import e2e_lm, lm_kernels
    cfg = e2e_lm.LMConfig(d_model=128, n_heads=3, d_head=64)
    op = e2e_lm.blhd_kernel(e2e_lm.operator_cfg(), 64)
    blk = _block(cfg, op).cuda()
    x = torch.randn(2, 192, 128, device="cuda", requires_grad=True)
    kinds = (e2e_lm.Dense, e2e_lm.CausalDepthwiseConv, e2e_lm.RMSNorm)
    assert lm_kernels.usable(blk, x, *kinds)
    leaves = [x] + list(blk.parameters())
    w = torch.randn(2, 192, 128, device="cuda")
    got = [blk(x)] + list(torch.autograd.grad(blk(x), leaves, w))
    blk.kernel_fn = lambda *a: op(*a)          # another mixer: the module forward
    assert not lm_kernels.usable(blk, x, *kinds)
    want = [blk(x)] + list(torch.autograd.grad(blk(x), leaves, w))
    for a, b in zip(got, want):
        assert a.is_contiguous() and rel_l2(a, b) <= 2e-5
    y = torch.randn(1, 8, 128, device="cuda", requires_grad=True)
    sc = torch.rand(128, device="cuda", requires_grad=True)
    for f in (lm_kernels._RmsNorm.apply, lm_kernels.rms_ref):
        g, = torch.autograd.grad(f(y, sc).square().sum(), y, create_graph=True)
        h = torch.autograd.grad(g.square().sum(), (y, sc))
        if f is lm_kernels.rms_ref:
            assert all(rel_l2(a, b) <= 1e-5 for a, b in zip(first, h))
        first = h


def test_module_forward_stays_in_charge():
    """CPU tensors, hooks, replaced submodules and misaligned or other-dtype inputs."""
    from atomic_gdn2 import e2e_lm, lm_kernels
    cfg = e2e_lm.LMConfig(d_model=64, n_heads=1, d_head=64)
    op = e2e_lm.blhd_kernel(e2e_lm.operator_cfg(), 64)
    kinds = (e2e_lm.Dense, e2e_lm.CausalDepthwiseConv, e2e_lm.RMSNorm)
    assert not lm_kernels.usable(_block(cfg, op), torch.zeros(1, 64, 64), *kinds)
    # the remaining conditions with the device test planted away
    real = lm_kernels._usable_input
    lm_kernels._usable_input = lambda x: True
    try:
        x = torch.zeros(1, 64, 64)
        assert lm_kernels.usable(_block(cfg, op), x, *kinds)
        assert not lm_kernels.usable(_block(cfg, lambda *a: a[0]), x, *kinds)
        b = _block(cfg, op)
        b.k_conv.register_forward_hook(lambda *a: None)
        assert not lm_kernels.usable(b, x, *kinds)
        b = _block(cfg, op)
        b.q_proj = torch.nn.Linear(64, 64, bias=False)
        assert not lm_kernels.usable(b, x, *kinds)
        b = _block(cfg, op)
        b.mlp_norm.eps = 1e-5
        assert not lm_kernels.usable(b, x, *kinds)
        assert not lm_kernels.usable(_block(cfg, op).double(), x, *kinds)
        assert not lm_kernels.usable(_block(dataclasses.replace(cfg, d_conv=3), op), x, *kinds)
        flat = torch.zeros(65)
        b = _block(cfg, op)
        b.mlp_norm.scale = torch.nn.Parameter(flat[1:])
        assert not lm_kernels.usable(b, x, *kinds)
        b = _block(cfg, op)
        del b.mlp_norm.scale                   # a plain tensor in a parameter's place, of another shape
        b.mlp_norm.scale = torch.zeros(32)
        assert not lm_kernels.usable(b, x, *kinds)
    finally:
        lm_kernels._usable_input = real


def test_a_wrapped_mixer_keeps_the_module_forward():
    """A mixer built around the operator is another mixer, also where functools.wraps has copied the
    operator's attributes: its body runs."""
    from atomic_gdn2 import e2e_lm, lm_kernels
    cfg = e2e_lm.LMConfig(d_model=64, n_heads=1, d_head=64)
    op = e2e_lm.blhd_kernel(e2e_lm.operator_cfg(), 64)

    @functools.wraps(op)
    def half(*a):
        return 0.5 * op(*a)

    kinds = (e2e_lm.Dense, e2e_lm.CausalDepthwiseConv, e2e_lm.RMSNorm)
    real = lm_kernels._usable_input
    lm_kernels._usable_input = lambda x: True           # the device test planted away
    try:
        x = torch.zeros(1, 64, 64)
        assert lm_kernels.usable(_block(cfg, op), x, *kinds)
        assert not lm_kernels.usable(_block(cfg, half), x, *kinds)
        assert not lm_kernels.usable(_block(cfg, functools.partial(op)), x, *kinds)
    finally:
        lm_kernels._usable_input = real


def test_a_patched_submodule_keeps_the_module_forward(monkeypatch):
    """A submodule whose forward was replaced on the instance or on its class, or that was taken out
    and replaced by a plain callable, runs as the program has it."""
    from atomic_gdn2 import e2e_lm, lm_kernels
    cfg = e2e_lm.LMConfig(d_model=64, n_heads=1, d_head=64)
    op = e2e_lm.blhd_kernel(e2e_lm.operator_cfg(), 64)
    kinds = (e2e_lm.Dense, e2e_lm.CausalDepthwiseConv, e2e_lm.RMSNorm)
    monkeypatch.setattr(lm_kernels, "_usable_input", lambda x: True)        # the device test planted away
    x = torch.zeros(1, 64, 64)
    for name in ("q_proj", "v_conv", "mlp_norm"):
        b = _block(cfg, op)
        assert lm_kernels.usable(b, x, *kinds)
        m = getattr(b, name)
        plain = m.forward
        m.forward = lambda y: 2.0 * plain(y)
        assert not lm_kernels.usable(b, x, *kinds)
        b = _block(cfg, op)
        delattr(b, name)
        setattr(b, name, lambda y: y)
        assert not lm_kernels.usable(b, x, *kinds)
        with monkeypatch.context() as mp:
            cls = type(m)
            f = cls.forward
            mp.setattr(cls, "forward", lambda self, y: 2.0 * f(self, y))
            assert not lm_kernels.usable(_block(cfg, op), x, *kinds)
            assert name != "mlp_norm" or not lm_kernels.norm_usable(_block(cfg, op).mlp_norm, x, e2e_lm.RMSNorm)


@pytest.mark.gpu
@pytest.mark.parametrize("B,L", [(1, 64), (1, 448), (1, 512), (2, 640), (1, 4032), (4, 2048)])   # parts: few rows, batched, accumulated
def test_block_as_exact_as_the_module_forward(B, L):
    """The block's output, dx and matrix gradients against float64 torch operations: the merged products
    leave none further off than a product per matrix does.  5 % is left for the element-wise steps'
    rounding, and 1 / sqrt(rows) for its spread: rounding that a row shares (the norms' factors, the
    decay) makes an error's norm one of about as many independent values, which varies by
    1 / sqrt(2 rows) from one evaluation to another.  dx as whole sums over all columns is 29 % off from
    1280 rows on, the narrow matrix as columns of the wide product 15 %."""
    _need_gpu()
    import sys
    from pathlib import Path
    sys.path.insert(0, str(Path(__file__).resolve().parents[1]))
    from oracle.gdn2_oracle import OracleCfg, forward_ref_blhd
    from atomic_gdn2 import e2e_lm
    cfg, opc = e2e_lm.LMConfig(), e2e_lm.operator_cfg()
    op, ocfg = e2e_lm.blhd_kernel(opc, cfg.d_head), OracleCfg.from_cfg(opc)
    oracle = lambda *a: forward_ref_blhd(*(t.cpu() for t in a), cfg.d_head ** -0.5, None, ocfg)[0].cuda()  # noqa: E731
    blk = _block(cfg, op).cuda()
    gen = torch.Generator(device="cuda").manual_seed(L)
    x = torch.randn(B, L, cfg.d_model, generator=gen, device="cuda").requires_grad_(True)
    dy = torch.randn(B, L, cfg.d_model, generator=gen, device="cuda")
    names = ["x"] + [n for n, _ in blk.named_parameters()]

    def run(m, x, dy):
        y = m(x)
        return [y.detach()] + list(torch.autograd.grad(y, [x] + list(m.parameters()), dy))

    got = run(blk, x, dy)
    blk.kernel_fn = lambda *a: op(*a)                    # another mixer: the module forward
    want = run(blk, x, dy)
    blk64 = e2e_lm.GDN2Block(cfg, oracle).cuda().double()
    blk64.load_state_dict({n: p.double() for n, p in blk.state_dict().items()})
    exact = run(blk64, x.detach().double().requires_grad_(True), dy.double())
    for n, g, w, e in zip(["y"] + names, got, want, exact):
        if n in ("y", "x") or n.endswith("weight") and "conv" not in n:
            assert rel_l2(g, e) <= (1.05 + (B * L) ** -0.5) * rel_l2(w, e), (n, rel_l2(g, e), rel_l2(w, e))


@pytest.mark.gpu
def test_gradients_have_storages_of_their_own():
    _need_gpu()
    from atomic_gdn2 import e2e_lm
    cfg = e2e_lm.LMConfig(d_model=128, n_heads=3, d_head=64, n_layers=2)
    model = e2e_lm.make_lm(cfg, seed=0)
    e2e_lm.lm_loss(model, e2e_lm.synthetic_tokens(cfg, batch=2, length=128)).backward()
    for n, p in model.named_parameters():
        assert p.grad.shape == p.shape and p.grad.is_contiguous(), n
        assert p.grad.untyped_storage().nbytes() == 4 * p.numel(), n
    assert len({p.grad.data_ptr() for p in model.parameters()}) == len(list(model.parameters()))
