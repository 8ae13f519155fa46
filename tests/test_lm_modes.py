"""The language-model block under function transforms, forward-mode differentiation, dispatch modes and
tracing: the module forward, whose operations these see, runs there."""
import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode


def _block(device, mixer=None):
    from atomic_gdn2 import e2e_lm
    cfg = e2e_lm.LMConfig(d_model=64, n_heads=1, d_head=64)
    torch.manual_seed(0)
    mixer = mixer or e2e_lm.blhd_kernel(e2e_lm.operator_cfg(), 64)
    return e2e_lm.GDN2Block(cfg, mixer).to(device).requires_grad_(False)


def _mix(q, k, v, w, b, g):
    return v * w + q * k * b * torch.exp(g)


BEHIND = ("out_proj.weight", "mlp_norm.scale", "down_proj.weight")     # weights the operator does not see


def _loss(blk, x):
    rest = {n: p for n, p in blk.named_parameters() if n not in BEHIND}
    return lambda ws: torch.func.functional_call(blk, {**rest, **ws}, (x,)).square().sum()


def _check_transforms(blk, x, transforms):
    ws = {n: p.detach() for n, p in blk.named_parameters() if n in BEHIND}
    loss = _loss(blk, x)
    leaves = {n: w.clone().requires_grad_(True) for n, w in ws.items()}
    want = dict(zip(leaves, torch.autograd.grad(loss(leaves), list(leaves.values()))))
    for n, g in torch.func.grad(loss)(ws).items() if "grad" in transforms else ():
        assert torch.allclose(g, want[n], rtol=1e-4, atol=1e-4 * float(want[n].abs().max())), n
    both = torch.func.vmap(loss)({n: torch.stack([w, 2.0 * w]) for n, w in ws.items()})
    assert torch.allclose(both[0], loss(ws), rtol=1e-4)
    dirs = {n: torch.ones_like(w) for n, w in ws.items()}
    slope = sum(float((want[n] * dirs[n]).sum()) for n in ws)
    if "jvp" in transforms:
        assert abs(float(torch.func.jvp(loss, (ws,), (dirs,))[1]) - slope) <= 1e-3 * abs(slope)
    with torch.autograd.forward_ad.dual_level():
        duals = {n: torch.autograd.forward_ad.make_dual(w, dirs[n]) for n, w in ws.items()}
        tangent = torch.autograd.forward_ad.unpack_dual(loss(duals)).tangent
    assert abs(float(tangent) - slope) <= 1e-3 * abs(slope)


def test_transforms_over_the_weights_behind_the_operator(monkeypatch):
    """On the CPU, with the device test planted away wherever no transform is active."""
    from atomic_gdn2 import e2e_lm, lm_kernels
    lm_kernels.register_operator(_mix, _mix)
    blk, x = _block("cpu", _mix), torch.randn(2, 64, 64)
    kinds = (e2e_lm.Dense, e2e_lm.CausalDepthwiseConv, e2e_lm.RMSNorm)
    real = lm_kernels._usable_input
    planted = lambda y: True if torch._C._functorch.peek_interpreter_stack() is not None else real(y)  # noqa: E731
    monkeypatch.setattr(lm_kernels, "_usable_input", planted)
    _check_transforms(blk, x, ("grad", "jvp"))
    monkeypatch.setattr(lm_kernels, "_usable_input", lambda y: True)
    ok = lambda: lm_kernels.usable(blk, x, *kinds) and lm_kernels.norm_usable(blk.mlp_norm, x, e2e_lm.RMSNorm)  # noqa: E731
    either = lambda: lm_kernels.usable(blk, x, *kinds) or lm_kernels.norm_usable(blk.mlp_norm, x, e2e_lm.RMSNorm)  # noqa: E731
    assert ok()
    with torch.device("cpu"):                  # a default device is no reason
        assert ok()
    with torch.autograd.forward_ad.dual_level():
        assert not either()

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, f, types, args=(), kwargs=None):
            return f(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, f, types, args=(), kwargs=None):
            return f(*args, **(kwargs or {}))

    for mode in (Dispatch(), Function()):
        with mode:
            assert not either()
    seen = []
    torch.jit.trace(lambda y: (seen.append(either()), y + 1)[1], torch.zeros(1), check_trace=False)
    assert seen == [False]
    compiled = []

    @torch.compile(backend="eager")
    def f(y):
        return y + (1 if lm_kernels._plain_mode() else 2)

    compiled.append(float(f(torch.zeros(1))))
    assert compiled == [2.0]


@pytest.mark.gpu
def test_transforms_on_the_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")
    # (func.grad and func.jvp wrap every tensor formed inside them, the operator's outputs too: refused)
    _check_transforms(_block("cuda"), torch.randn(2, 64, 64, device="cuda"), ())
