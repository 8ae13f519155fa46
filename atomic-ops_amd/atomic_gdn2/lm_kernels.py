"""The language-model block of ``e2e_lm`` on the HIP passes of ``csrc/gdn2_lm.hip``.

``block_forward`` computes what ``GDN2Block.forward`` computes, with the element-wise chains
between the matrix products in one kernel each and the products that share an input as one GEMM:

* ``_PreMix``   x -> one GEMM with [Wq | Wk | Wv | We | Ww | Wo | Wd] -> q, k, v, w, b, g head-major,
  the layout the operator reads, and the output gate's logits;
* ``_PostMix``  the operator's o -> RMS norm, SiLU gate, output projection, residual;
* ``_Mlp``      RMS norm, gate / up as one GEMM, SiLU(gate) * up, down projection, residual.

Each is one autograd node whose backward runs the matching backward kernels.  A backward that is
itself to be differentiated (``create_graph``) recomputes the step from ``_premix_ref`` /
``_postmix_ref`` / ``_mlp_ref``, the same in torch operations; the operator between them is
differentiable once, and a second derivative through it raises.

``usable`` says where this path stands in for the module's own forward: float32 on the GPU, the
block's own submodule types without hooks, the HIP operator as the mixer.  Everywhere else (the CPU,
other dtypes, autocast, function transforms, forward mode, dispatch modes, tracing, hooked, patched or
replaced submodules, another mixer) the module forward runs.
"""
from __future__ import annotations

import ctypes
import types
import weakref

import torch
import torch.nn.functional as F
import torch.overrides
import torch.utils._device

from . import _lib

_i32, _f32c, _vp = ctypes.c_int32, ctypes.c_float, ctypes.c_void_p
_EPS = 1e-6
_MAX_C = 1024           # widest row of the RMS kernels


class _PremixArgs(ctypes.Structure):
    _fields_ = [("B", _i32), ("L", _i32), ("H", _i32), ("D", _i32), ("ldy", _i32), ("g_max", _f32c), ("y", _vp),
                ("conv_w", _vp * 3), ("conv_b", _vp * 3), ("gate_b", _vp * 2), ("decay_b", _vp), ("decay_a", _vp),
                ("out", _vp * 6), ("og", _vp)]


class _RmsArgs(ctypes.Structure):
    _fields_ = [("rows", _i32), ("C", _i32), ("L", _i32), ("D", _i32)] + [
        (n, _vp) for n in ("x", "gate", "scale", "dy", "res", "y", "dx", "dgate", "part", "dscale")]


def _addr(t):
    return None if t is None else t.data_ptr()


def _dense(t):
    """t as the kernels read it: contiguous, 16-byte aligned."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _save(ctx, *ts):
    ctx.save_for_backward(*ts)
    ctx.forms = _lib.bind().forms(ts)


def _saved(ctx):
    """The saved tensors in the form they were saved in."""
    ts = ctx.saved_tensors
    differ = _lib.bind().differ(ctx.forms, ts)
    if not differ:
        return ts
    return tuple(t if f is None else _dense(_lib.restored(t, *f)) for t, f in zip(ts, differ))


def _call(name, dev, *args):
    fn = getattr(_lib.lib(), name)
    with torch.cuda.device(dev):
        _lib.check(fn(*args, _lib.stream_handle(dev)), name)


def _rms(x, scale, gate=None, heads=None):
    """RMS norm of the rows of x (N, C), or of the head-major o with heads = (L, D) and a gate."""
    rows, C = (x.shape[0], x.shape[1]) if gate is None else (gate.shape[0], gate.shape[1])
    y = torch.empty((rows, C), dtype=torch.float32, device=x.device)
    L, D = heads or (0, 0)
    a = _RmsArgs(rows, C, L, D, _addr(x), _addr(gate), _addr(scale), None, None, _addr(y), None, None, None, None)
    _call("gdn2_lm_rms_fwd", x.device, ctypes.byref(a))
    return y


def _rms_bwd(x, scale, dy, gate=None, heads=None, res=None):
    rows, C = dy.shape
    dev = x.device
    dx, dscale = torch.empty_like(x), torch.empty_like(scale)
    dgate = None if gate is None else torch.empty_like(gate)
    part = torch.empty(_lib.lib().gdn2_lm_rms_workspace_bytes(rows, C) // 4, dtype=torch.float32, device=dev)
    L, D = heads or (0, 0)
    a = _RmsArgs(rows, C, L, D, _addr(x), _addr(gate), _addr(scale), _addr(dy), _addr(res), None, _addr(dx),
                 _addr(dgate), _addr(part), _addr(dscale))
    _call("gdn2_lm_rms_bwd", dev, ctypes.byref(a))
    return dx, dscale, dgate


def _swiglu(gu, d_act=None):
    rows, M2 = gu.shape
    out = torch.empty((rows, M2 // 2 if d_act is None else M2), dtype=torch.float32, device=gu.device)
    _call("gdn2_lm_swiglu", gu.device, _addr(gu), _addr(d_act), _addr(out), rows, M2 // 2)
    return out


def _columns(split, parts, wide):
    n, rows = len(parts), wide.shape[0]
    ptrs = (_vp * n)(*(t.data_ptr() for t in parts))
    widths = (_i32 * n)(*(t.numel() // rows for t in parts))
    _call("gdn2_lm_columns", wide.device, int(split), ptrs, widths, n, _addr(wide), rows, wide.shape[1])


def _gather(parts, ld):
    """The matrices side by side, zero-padded to ld columns."""
    wide = torch.empty((parts[0].shape[0], ld), dtype=torch.float32, device=parts[0].device)
    _columns(0, parts, wide)
    return wide


def _scatter(wide, like):
    """wide back into matrices of the shapes of ``like`` (vectors from a wide of one row), each with a
    storage of its own: they become parameters' gradients, which a program keeps, saves or frees singly."""
    out = [torch.empty(t.shape, dtype=torch.float32, device=wide.device) for t in like]
    _columns(1, out, wide)
    return out


def _weight_grad(x, dy):
    """x^T dy over the rows, in two halves from 8192 rows on: the library's kernels for these shapes
    leave one long reduction at 100 TFLOP/s, two batched halves run at 126 (512 x 4672: 16384 rows
    778 -> 614 us, 8192 378 -> 315, 4096 187 and 188; 768 x 512: 124 -> 105, 63 -> 59, 36 and 34).  The
    MLP's products stay whole (512 x 2048: 16384 rows 254 and 246, 8192 126 and 124; 1024 x 512: 135 and
    129, 67 and 70)."""
    n = x.shape[0]
    if n < 8192 or n % 2:
        return x.t() @ dy
    halves = torch.bmm(x.view(2, n // 2, -1).transpose(1, 2), dy.view(2, n // 2, -1))
    return halves[0] + halves[1]


def _narrow_weight_grad(x, dy):
    """x^T dy for a dy of a few columns.  The library splits such a product's long sum, which beside
    the wide ones it does not (16384 rows, 512 x 6: 11.7e-7 of the result, as columns of the wide
    product 15.7e-7 in halves, 22e-7 whole), but not over enough of the chip: 58 us.  Sixteen batched
    parts from 4096 rows on: 3.0e-7, about 10 us."""
    n = x.shape[0]
    if n < 4096 or n % 16:
        return x.t() @ dy
    return torch.bmm(x.view(16, n // 16, -1).transpose(1, 2), dy.view(16, n // 16, -1)).sum(0)


def _input_grad(dy, wide, parts, parts_few):
    """dy wide^T with the sum over the columns in parts.  Rounding errors add up along a sum: as whole
    sums over 4672 and 2048 columns (12.2e-7 and 8.1e-7 of the result) these two products took the
    block's dx from 6.6e-7 of the exact one, where a product per matrix has it, to 8.5e-7 (B4 L2048).
    Halves of the one and quarters of the other (8.6e-7, 4.1e-7; the MLP's weighs more in dx) keep it at
    6.5e-7, in less time than one part per matrix (601 + 251 us at 16384 rows, 253 + 103 at 4864):
    from 8192 rows on the parts accumulate into the result one after the other (16384 rows: 525 ->
    539 us and 237 -> 273), below they are one batched product and a sum (4864: 200 -> 193 and
    89 -> 99).  For few rows the library splits a single matrix's sum by itself (up to 256 rows:
    2.6e-7, 2.9e-7), but not a batch's: parts_few below 512."""
    N, K = dy.shape
    m = parts if N >= 512 else parts_few
    w = K // m
    if N >= 8192:
        dx = dy[:, :w] @ wide[:, :w].t()
        for i in range(w, K, w):
            dx.addmm_(dy[:, i:i + w], wide[:, i:i + w].t())
        return dx
    return torch.bmm(dy.view(N, m, w).transpose(0, 1), wide.view(-1, m, w).permute(1, 2, 0)).sum(0)


def _vjp_through(ref, inputs, needs, grads):
    """Gradients of ref(*inputs) for a backward that is itself differentiated.  They are taken at
    aliases of the inputs: an input may be computed from another one (the operator's o and the
    gate's logits from x) or appear twice (a tied weight), and each gradient is this node's own
    share, without the paths that lie outside it."""
    with torch.enable_grad():
        inputs = [x.view_as(x) for x in inputs]
        outs = ref(*inputs)
        outs = outs if isinstance(outs, tuple) else (outs,)
        pairs = [(o, g) for o, g in zip(outs, grads) if g is not None and o.requires_grad]
        wrt = [x for x, n in zip(inputs, needs) if n]
        got = iter(torch.autograd.grad([o for o, _ in pairs], wrt, [g for _, g in pairs], create_graph=True,
                                       allow_unused=True))
    return tuple(next(got) if n else None for n in needs)


# ------------------------------------------------------------------------------------------
# the steps in torch operations
# ------------------------------------------------------------------------------------------

def conv_ref(x, weight, bias):
    """Causal depthwise convolution of (B, L, C): K shifted multiply-adds."""
    K = weight.shape[1]
    y = torch.addcmul(bias, x, weight[:, K - 1])
    for s in range(1, K):
        y = torch.addcmul(y, F.pad(x[:, :-s], (0, 0, s, 0)), weight[:, K - 1 - s])
    return y


def rms_ref(x, scale, eps=_EPS):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * scale


def decay_ref(logits, decay_a, g_max):
    """Per-head log-decay (B, L, H) of the decay logits."""
    ldh = -torch.exp(decay_a.clamp(-20, 20)) * F.softplus(logits)
    ld = torch.nan_to_num(ldh, nan=0.0, posinf=0.0, neginf=-20.0)
    return -ld.abs().clamp(max=g_max)


def _premix_ref(H, D, g_max):
    def ref(x, wq, wk, wv, we, ww, wo, wd, cqw, cqb, ckw, ckb, cvw, cvb, be, bw, bd, da):
        B, L, _ = x.shape
        heads = lambda y: y.reshape(B, L, H, D).transpose(1, 2)  # noqa: E731
        q, k, v = (heads(F.silu(conv_ref(x @ w, cw, cb)))
                   for w, cw, cb in ((wq, cqw, cqb), (wk, ckw, ckb), (wv, cvw, cvb)))
        q, k = (y * torch.rsqrt((y * y).sum(-1, keepdim=True) + _EPS) for y in (q, k))
        b, w = heads(torch.sigmoid(x @ we + be)), heads(torch.sigmoid(x @ ww + bw))
        g = decay_ref(x @ wd + bd, da, g_max).transpose(1, 2).unsqueeze(-1).expand(B, H, L, D)
        return q, k, v.clamp(-50.0, 50.0), w, b, g, (x @ wo).reshape(B * L, H * D)
    return ref


def _postmix_ref(o, og, x, scale, wo):
    B, H, L, D = o.shape
    z = rms_ref(o.transpose(1, 2).reshape(B * L, H * D), scale) * F.silu(og)
    return x + (z @ wo).reshape(x.shape)


def _mlp_ref(x, scale, wg, wu, wd):
    h = rms_ref(x, scale)
    return x + (F.silu(h @ wg) * (h @ wu)) @ wd


# ------------------------------------------------------------------------------------------
# the autograd nodes
# ------------------------------------------------------------------------------------------

class _PreMix(torch.autograd.Function):
    """(x, Wq, Wk, Wv, We, Ww, Wo, Wd, conv taps and biases of q, k, v, be, bw, bd, decay_a) ->
    q, k, v, w, b, g (B, H, L, D), output-gate logits (B L, C)."""

    @staticmethod
    def forward(ctx, H, D, g_max, x, *ps):
        B, L, d = x.shape
        C, dev = H * D, x.device
        ws = ps[:7]
        ldy = -(-(6 * C + H) // 64) * 64
        wide = _gather(ws, ldy)
        y = x.reshape(B * L, d) @ wide
        outs = [torch.empty((B, H, L, D), dtype=torch.float32, device=dev) for _ in range(6)]
        og = torch.empty((B * L, C), dtype=torch.float32, device=dev)
        a = _PreMix._args(H, D, g_max, x, ps, y, outs, og)
        _call("gdn2_lm_premix_fwd", dev, ctypes.byref(a))
        ctx.dims = (H, D, g_max)
        _save(ctx, x, *ps, wide, y, *outs, og)
        return (*outs, og)

    @staticmethod
    def _args(H, D, g_max, x, ps, y, outs, og):
        cqw, cqb, ckw, ckb, cvw, cvb, be, bw, bd, da = (t.data_ptr() for t in ps[7:])
        return _PremixArgs(x.shape[0], x.shape[1], H, D, y.shape[1], float(g_max), y.data_ptr(), (_vp * 3)(cqw, ckw, cvw),
                           (_vp * 3)(cqb, ckb, cvb), (_vp * 2)(be, bw), bd, da, (_vp * 6)(*(t.data_ptr() for t in outs)),
                           og.data_ptr())

    @staticmethod
    def backward(ctx, *gs):
        H, D, g_max = ctx.dims
        saved = _saved(ctx)
        x, ps, wide, y, outs, og = saved[0], saved[1:18], saved[18], saved[19], saved[20:26], saved[26]
        if torch.is_grad_enabled():
            return (None, None, None) + _vjp_through(_premix_ref(H, D, g_max), (x,) + ps, ctx.needs_input_grad[3:], gs)
        B, L, d = x.shape
        C, dev, N = H * D, x.device, x.shape[0] * x.shape[1]
        like = list(outs) + [og]
        ds = [torch.zeros_like(t) if g is None else _dense(g) for g, t in zip(gs, like)]
        dy = torch.empty_like(y)
        dparam = torch.empty(17 * C + 2 * H, dtype=torch.float32, device=dev)
        ws = torch.empty(_lib.lib().gdn2_lm_premix_workspace_bytes(B, L, H, D), dtype=torch.uint8, device=dev)
        a = _PreMix._args(H, D, g_max, x, ps, y, outs, og)
        _call("gdn2_lm_premix_bwd", dev, ctypes.byref(a), (_vp * 6)(*(t.data_ptr() for t in ds[:6])), _addr(ds[6]),
              _addr(dy), _addr(dparam), _addr(ws))
        need = ctx.needs_input_grad[3:]
        dx = _input_grad(dy, wide, 2, 32).reshape(B, L, d) if need[0] else None
        x2, dws = x.reshape(N, d), [None] * 7
        if any(need[1:7]):
            dws[:6] = _scatter(_weight_grad(x2, dy[:, :6 * C]), ps[:6])
        if need[7]:
            dws[6] = _narrow_weight_grad(x2, dy[:, 6 * C:6 * C + H])
        dps = _scatter(dparam.view(1, -1), ps[7:]) if any(need[8:]) else [None] * 10
        return (None, None, None) + tuple(g if n else None for g, n in zip([dx, *dws, *dps], need))


class _PostMix(torch.autograd.Function):
    """(o (B, H, L, D), output-gate logits, x, norm scale, Wout) -> x + (rms(o) scale silu(og)) Wout."""

    @staticmethod
    def forward(ctx, o, og, x, scale, wo):
        B, H, L, D = o.shape
        z = _rms(o, scale, og, (L, D))
        _save(ctx, o, og, x, scale, wo, z)
        return torch.addmm(x.reshape(B * L, -1), z, wo).reshape(x.shape)

    @staticmethod
    def backward(ctx, dy):
        o, og, x, scale, wo, z = _saved(ctx)
        if torch.is_grad_enabled():
            return _vjp_through(_postmix_ref, (o, og, x, scale, wo), ctx.needs_input_grad, (dy,))
        need = ctx.needs_input_grad
        B, H, L, D = o.shape
        d2 = dy.reshape(B * L, -1)
        do = dog = dscale = None
        if need[0] or need[1] or need[3]:
            do, dscale, dog = _rms_bwd(o, scale, d2 @ wo.t(), og, (L, D))
        dwo = _weight_grad(z, d2.contiguous()) if need[4] else None
        return tuple(g if n else None for g, n in zip((do, dog, dy, dscale, dwo), need))


class _Mlp(torch.autograd.Function):
    """(x, norm scale, Wgate, Wup, Wdown) -> x + (silu(h Wgate) (h Wup)) Wdown, h = rms(x) scale."""

    @staticmethod
    def forward(ctx, x, scale, wg, wu, wd):
        x2 = x.reshape(-1, x.shape[-1])
        h = _rms(x2, scale)
        wide = _gather((wg, wu), 2 * wg.shape[1])
        gu = h @ wide
        act = _swiglu(gu)
        _save(ctx, x, scale, wg, wu, wd, h, wide, gu, act)
        return torch.addmm(x2, act, wd).reshape(x.shape)

    @staticmethod
    def backward(ctx, dy):
        x, scale, wg, wu, wd, h, wide, gu, act = _saved(ctx)
        if torch.is_grad_enabled():
            return _vjp_through(_mlp_ref, (x, scale, wg, wu, wd), ctx.needs_input_grad, (dy,))
        need = ctx.needs_input_grad
        d2 = _dense(dy.reshape(-1, dy.shape[-1]))
        dgu = _swiglu(gu, d2 @ wd.t())
        dwd = act.t() @ d2 if need[4] else None
        dwg, dwu = _scatter(h.t() @ dgu, (wg, wu)) if need[2] or need[3] else (None, None)
        dx, dscale, _ = _rms_bwd(x.reshape(d2.shape), scale, _input_grad(dgu, wide, 4, 8), res=d2)
        return tuple(g if n else None for g, n in zip((dx.reshape(x.shape), dscale, dwg, dwu, dwd), need))


class _RmsNorm(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, scale):
        _save(ctx, x, scale)
        return _rms(x.reshape(-1, x.shape[-1]), scale).reshape(x.shape)

    @staticmethod
    def backward(ctx, dy):
        x, scale = _saved(ctx)
        if torch.is_grad_enabled():
            return _vjp_through(rms_ref, (x, scale), ctx.needs_input_grad, (dy,))
        d2 = _dense(dy.reshape(-1, dy.shape[-1]))
        dx, dscale, _ = _rms_bwd(x.reshape(d2.shape), scale, d2)
        return dx.reshape(x.shape), dscale


# ------------------------------------------------------------------------------------------
# the block
# ------------------------------------------------------------------------------------------

_HOOKS = ("_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks")
_DENSE = ("q_proj", "k_proj", "v_proj", "erase_gate", "write_gate", "out_gate", "decay_proj", "out_proj", "gate_proj",
          "up_proj", "down_proj")
_CONV = ("q_conv", "k_conv", "v_conv")
_NORM = ("mixer_out_norm", "mlp_norm")
_BIASED = ("erase_gate", "write_gate", "decay_proj")


def _ready(t, dev):
    return (t.device == dev and t.dtype == torch.float32 and t.is_contiguous() and t.data_ptr() % 16 == 0
            and t.numel() > 0)


_FORWARDS = {}          # module class -> its own forward


def register_modules(*classes):
    """Declare the module classes a block is built of, with the forwards that block_forward computes."""
    _FORWARDS.update((c, c.forward) for c in classes)


def _plain(m, cls):
    return (type(m) is cls and cls.forward is _FORWARDS.get(cls) and "forward" not in m.__dict__
            and not any(getattr(m, h) for h in _HOOKS))


def _plain_mode():
    """Whether a node of this module is an ordinary call here.  Function transforms and forward mode
    have no rules for the nodes, and dispatch modes, function modes and tracers are to see the block's
    operations; a default device (itself a function mode) is no reason."""
    return not (torch.compiler.is_compiling()
                or torch._C._functorch.peek_interpreter_stack() is not None
                or torch.autograd.forward_ad._current_level >= 0
                or torch._C._len_torch_dispatch_stack() > 0
                or torch._C._get_tracing_state() is not None
                or (torch._C._len_torch_function_stack() > 0
                    and any(type(m) is not torch.utils._device.DeviceContext
                            for m in torch.overrides._get_current_function_mode_stack())))


def _usable_input(x):
    return (x.is_cuda and type(x) in (torch.Tensor, torch.nn.Parameter) and _ready(x, x.device)
            and x.shape[-1] % 4 == 0 and x.shape[-1] <= _MAX_C and not torch.is_autocast_enabled("cuda")
            and not torch.nn.modules.module._has_any_global_hook())


_OPERATORS = weakref.WeakKeyDictionary()    # a (B, L, H, D) mixer -> the operator it stands for


def register_operator(mixer, operator):
    """Declare that the function ``mixer`` of (B, L, H, D) tensors is the HIP operator ``operator`` of
    head-major ones, so that a block may call the latter.  Kept by the function's identity: a wrapper
    around the mixer is another mixer, whatever attributes it copied."""
    _OPERATORS[mixer] = operator


def operator_of(mixer):
    """The head-major operator that mixer was registered for, or None."""
    return _OPERATORS.get(mixer) if type(mixer) is types.FunctionType else None


def usable(block, x, dense, conv, norm):
    """Whether block_forward stands for block.forward(x); dense, conv, norm: the module types that
    the block is built of."""
    return block_tensors(block, x, dense, conv, norm) is not None


def block_tensors(block, x, dense, conv, norm):
    """The block's weights as block_forward takes them, or None where the module forward runs."""
    c = block.cfg
    if operator_of(block.kernel_fn) is None or not (_plain_mode() and x.dim() == 3 and _usable_input(x)):
        return None
    if c.d_head not in (64, 128) or c.d_conv != 4 or c.proj_dim > _MAX_C or (c.mlp_mult * c.d_model) % 4:
        return None
    mods = block._modules
    if not (all(_plain(mods.get(n), dense) for n in _DENSE) and all(_plain(mods.get(n), conv) for n in _CONV)
            and all(_plain(mods.get(n), norm) and mods[n].eps == _EPS for n in _NORM)):
        return None
    if any((mods[n].bias is None) == (n in _BIASED) for n in _DENSE):
        return None
    d, p, H, M = c.d_model, c.proj_dim, c.n_heads, c.mlp_mult * c.d_model
    shapes = [(d, p)] * 6 + [(d, H)] + [(p, 4), (p,)] * 3 + [(p,)] * 2 + [(H,)] * 2 + [(p,), (p, d), (d,), (d, M), (d, M), (M, d)]
    if x.shape[-1] != d:
        return None
    ts = _tensors(block)
    if not all(type(t) in (torch.Tensor, torch.nn.Parameter) and t.shape == sh for t, sh in zip(ts, shapes)):
        return None
    return ts if _lib.bind().dense(ts, x) else None


def _tensors(m):
    """The block's weights in the order the three nodes take them (17, then 2, then 4)."""
    return (m.q_proj.weight, m.k_proj.weight, m.v_proj.weight, m.erase_gate.weight, m.write_gate.weight, m.out_gate.weight,
            m.decay_proj.weight, m.q_conv.weight, m.q_conv.bias, m.k_conv.weight, m.k_conv.bias, m.v_conv.weight,
            m.v_conv.bias, m.erase_gate.bias, m.write_gate.bias, m.decay_proj.bias, m.decay_a,
            m.mixer_out_norm.scale, m.out_proj.weight,
            m.mlp_norm.scale, m.gate_proj.weight, m.up_proj.weight, m.down_proj.weight)


def norm_usable(module, x, norm):
    return (_plain_mode() and _plain(module, norm) and module.eps == _EPS and _usable_input(x)
            and type(module.scale) in (torch.Tensor, torch.nn.Parameter) and module.scale.shape == x.shape[-1:]
            and _ready(module.scale, x.device))


def rms_norm(module, x):
    return _RmsNorm.apply(x, module.scale)


def block_forward(m, x, ws):
    c = m.cfg
    *ops, og = _PreMix.apply(c.n_heads, c.d_head, c.g_max, x, *ws[:17])
    o, _ = operator_of(m.kernel_fn)(*ops)
    x = _PostMix.apply(o, og, x, *ws[17:19])
    return _Mlp.apply(x, *ws[19:])
