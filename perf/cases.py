"""The work that programs using this framework have it do, as measured cases.

Six kinds of calls, each through the public entry points:

* ``decode``   one token of serving for a batch of sequences (``inference.decode_step``);
* ``prefill``  a prompt of any length, with document resets (``inference.chunk_forward_inference``);
* ``forward``  the operator without gradients, the state carried in (``make_blr_trainable``);
* ``grad``     the operator forward and backward (``make_blr_trainable`` under autograd);
* ``block``    one layer of the language model, forward and backward (``e2e_lm.GDN2Block``);
* ``lm``       the language model: logits, next-token loss and all gradients (``e2e_lm``).

Inputs follow the operator's benchmark distributions: q, k, w rows L2-normalised, v ~ N(0,1),
b = sigmoid(N), g = -0.1 softplus(N), scale 1/sqrt(D).
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "atomic-ops_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from atomic_gdn2 import make_blr_trainable, make_cfg  # noqa: E402
from atomic_gdn2 import e2e_lm  # noqa: E402
from atomic_gdn2.inference import chunk_forward_inference, decode_step  # noqa: E402

DEV = "cuda"


# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------

def listed():
    return [
        # one user's next token, as a single sequence is served: all latency
        {"name": "decode_b1h6", "kind": "decode", "B": 1, "H": 6, "D": 128, "dtype": "fp32", "fuse": False,
         "reset": False, "cap": False},
        # the serving batch of the inference benchmark, from raw projections (gates and norms formed
        # by the call), bf16 inputs and state, some rows starting a new document
        {"name": "decode_b8h16_bf16", "kind": "decode", "B": 8, "H": 16, "D": 128, "dtype": "bf16", "fuse": True,
         "reset": True, "cap": False},
        # a large serving batch: the state streams through the chip
        {"name": "decode_b64h16", "kind": "decode", "B": 64, "H": 16, "D": 128, "dtype": "fp32", "fuse": False,
         "reset": False, "cap": False},
        # packed documents of a length that is no multiple of the chunk
        {"name": "prefill_docs_b2h16_l3000", "kind": "prefill", "B": 2, "H": 16, "L": 3000, "D": 128,
         "dtype": "bf16", "state": "fp32", "docs": 4},
        # one segment of the long-context forward: bf16 inputs, the fp32 state carried in
        {"name": "forward_b8h16_l4096_bf16", "kind": "forward", "B": 8, "H": 16, "L": 4096, "D": 128,
         "dtype": "bf16", "h0": True},
        # one long sequence of a small model: few heads, many chunks
        {"name": "forward_b1h6_l8192", "kind": "forward", "B": 1, "H": 6, "L": 8192, "D": 128, "dtype": "fp32",
         "h0": False},
        # the smallest training call of the benchmark
        {"name": "grad_b1h2_l256", "kind": "grad", "B": 1, "H": 2, "L": 256, "D": 128, "cfg": "highest", "bs2": 32,
         "h0": False},
        # the headline gradient evaluation
        {"name": "grad_b4h6_l2048", "kind": "grad", "B": 4, "H": 6, "L": 2048, "D": 128, "cfg": "highest",
         "bs2": 32, "h0": False},
        # the default configuration (chunk 128, damped, bf16x3 backward) over two segments, few heads
        {"name": "grad_prod_b4h2_l4096", "kind": "grad", "B": 4, "H": 2, "L": 4096, "D": 128, "cfg": "prod",
         "bs2": 32, "h0": False},
        # the narrower head, odd counts, a carried-in state with its gradient
        {"name": "grad_b3h5_l1472_d64", "kind": "grad", "B": 3, "H": 5, "L": 1472, "D": 64, "cfg": "highest",
         "bs2": 16, "h0": True},
        # one layer of the language model in training
        {"name": "block_b4_l2048", "kind": "block", "B": 4, "L": 2048},
        # the benchmark language model's forward and backward
        {"name": "lm_b8_l2048", "kind": "lm", "B": 8, "L": 2048},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "prefill", "forward", "forward", "grad", "grad", "block", "lm"])
    D = rng.choice([64, 128, 128])
    if kind == "decode":
        return {"kind": kind, "B": _log_int(rng, 1, 64), "H": rng.randint(1, 16), "D": D,
                "dtype": rng.choice(["fp32", "bf16"]), "fuse": rng.random() < 0.5, "reset": rng.random() < 0.5,
                "cap": rng.random() < 0.25}
    if kind == "prefill":
        return {"kind": kind, "B": rng.randint(1, 4), "H": rng.randint(2, 16), "L": _log_int(rng, 70, 4096), "D": D,
                "dtype": rng.choice(["fp32", "bf16"]), "state": rng.choice(["fp32", "bf16"]),
                "docs": rng.choice([1, 2, 3, 5])}
    if kind == "forward":
        return {"kind": kind, "B": _log_int(rng, 1, 8), "H": rng.randint(1, 16), "L": 64 * _log_int(rng, 4, 128), "D": D,
                "dtype": rng.choice(["fp32", "bf16"]), "h0": rng.random() < 0.5}
    if kind == "grad":
        cfg = rng.choice(["highest", "highest", "bf16x3", "prod"])
        unit = 128 if cfg == "prod" else 64
        return {"kind": kind, "B": rng.randint(1, 4), "H": rng.randint(1, 6), "L": unit * _log_int(rng, 2, 4096 // unit),
                "D": D, "cfg": cfg, "bs2": rng.choice([16, 32, 32, 64]), "h0": rng.random() < 0.3}
    if kind == "block":
        return {"kind": kind, "B": rng.randint(1, 8), "L": 64 * _log_int(rng, 2, 32)}
    return {"kind": kind, "B": rng.randint(1, 4), "L": 64 * _log_int(rng, 2, 24)}


# ---------------------------------------------------------------------------------------------
# what the program has in hand
# ---------------------------------------------------------------------------------------------

def _dtype(name):
    return torch.bfloat16 if name == "bf16" else torch.float32


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEV)


def _unit(x):
    return x / torch.linalg.vector_norm(x, dim=-1, keepdim=True)


def _inputs(gen, shape):
    q, k, v, w, b, g = (_randn(gen, *shape) for _ in range(6))
    return [_unit(q), _unit(k), v, _unit(w), torch.sigmoid(b), -0.1 * F.softplus(g)]


def _state(gen, B, H, D):
    return 0.3 * _randn(gen, B, H, D, D)


def _highest(**kw):
    base = dict(bt=64, bc=32, score_bs=64, bs2=32, mb=8, wy_eps=0.0, dot_mode="highest", solve_dot_mode="highest",
                b3_dot_mode="highest")
    base.update(kw)
    return make_cfg(**base)


def _cfg(case):
    if case["cfg"] == "prod":
        return make_cfg(bs2=case["bs2"])
    if case["cfg"] == "bf16x3":
        return _highest(bs2=case["bs2"], dot_mode="bf16x3", solve_dot_mode="bf16x3", b3_dot_mode="bf16x3")
    return _highest(bs2=case["bs2"])


def _documents(case, seed):
    """(B, L) document ids that change at chunk starts only."""
    B, L = case["B"], case["L"]
    ids = torch.zeros(B, L, dtype=torch.int64)
    gen = torch.Generator().manual_seed(seed)
    for r in range(B):
        for c in torch.randint(1, max(2, L // 64), (case["docs"] - 1,), generator=gen).tolist():
            if 64 * c < L:
                ids[r, 64 * c:] += 1
    return ids.to(DEV)


def prepare(case, seed):
    kind, gen = case["kind"], _gen(seed)
    if kind == "decode":
        B, H, D = case["B"], case["H"], case["D"]
        dt = _dtype(case["dtype"])
        s = {"case": case, "scale": D ** -0.5, "state": _state(gen, B, H, D).to(dt)}
        if case["fuse"]:
            xs = [_randn(gen, B, H, D) for _ in range(6)]
            s["a_log"], s["dt_bias"] = 0.5 * _randn(gen, H) - 2.0, 0.5 * _randn(gen, D) - 1.0
        else:
            xs = _inputs(gen, (B, H, D))
            s["a_log"] = s["dt_bias"] = None
        s["xs"] = [x.to(dt) for x in xs]
        s["reset"] = (torch.rand(B, generator=gen, device=DEV) < 0.25).to(torch.int32) if case["reset"] else None
        s["tau"] = 30.0 if case["cap"] else None
        return s
    if kind == "prefill":
        B, H, L, D = (case[n] for n in "BHLD")
        return {"case": case, "scale": D ** -0.5, "xs": [x.to(_dtype(case["dtype"])) for x in _inputs(gen, (B, H, L, D))],
                "ids": _documents(case, seed), "cfg": _highest()}
    if kind in ("forward", "grad"):
        B, H, L, D = (case[n] for n in "BHLD")
        xs = _inputs(gen, (B, H, L, D))
        h0 = _state(gen, B, H, D) if case["h0"] else None
        s = {"case": case, "scale": D ** -0.5, "h0": h0}
        if kind == "forward":
            s["xs"] = [x.to(_dtype(case["dtype"])) for x in xs]
            s["fn"] = make_blr_trainable(_highest(), s["scale"])
            return s
        s["xs"] = [x.requires_grad_(True) for x in xs]
        if h0 is not None:
            h0.requires_grad_(True)
        # the cotangents that the layers above hand down
        s["do"], s["dh"] = 0.1 * _randn(gen, B, H, L, D), 0.1 * _randn(gen, B, H, D, D)
        s["fn"] = make_blr_trainable(_cfg(case), s["scale"])
        return s
    cfg = e2e_lm.LMConfig()
    if kind == "block":
        torch.manual_seed(seed)
        block = e2e_lm.GDN2Block(cfg, e2e_lm.blhd_kernel(e2e_lm.operator_cfg(), cfg.d_head)).to(DEV)
        x = _randn(gen, case["B"], case["L"], cfg.d_model).requires_grad_(True)
        return {"case": case, "block": block, "x": x, "dy": _randn(gen, case["B"], case["L"], cfg.d_model),
                "params": list(block.parameters())}
    model = e2e_lm.make_lm(cfg, device=DEV, seed=seed)
    return {"case": case, "model": model, "params": list(model.parameters()),
            "ids": e2e_lm.synthetic_tokens(cfg, batch=case["B"], length=case["L"], seed=seed, device=DEV)}


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        o, st = decode_step(*s["xs"], s["state"], s["scale"], reset=s["reset"], state_dtype=_dtype(case["dtype"]),
                            stability_tau=s["tau"], fuse_prologue=case["fuse"], a_log=s["a_log"],
                            dt_bias=s["dt_bias"])
        return {"o": o, "state": st}
    if kind == "prefill":
        o, h = chunk_forward_inference(*s["xs"], s["scale"], s["cfg"], segment_ids=s["ids"],
                                       state_dtype=_dtype(case["state"]))
        return {"o": o, "h": h}
    if kind == "forward":
        with torch.no_grad():
            o, h = s["fn"](*s["xs"], s["h0"])
        return {"o": o, "h": h}
    if kind == "grad":
        leaves = s["xs"] + ([s["h0"]] if s["h0"] is not None else [])
        o, h = s["fn"](*s["xs"], s["h0"])
        grads = torch.autograd.grad((o, h), leaves, (s["do"], s["dh"]))
        return {"o": o.detach(), "h": h.detach(), "grads": list(grads)}
    if kind == "block":
        y = s["block"](s["x"])
        grads = torch.autograd.grad(y, [s["x"]] + s["params"], s["dy"])
        return {"y": y.detach(), "grads": list(grads)}
    ids = s["ids"]
    logits = s["model"](ids)
    V = logits.shape[-1]
    loss = F.cross_entropy(logits[:, :-1].reshape(-1, V), ids[:, 1:].reshape(-1))
    grads = torch.autograd.grad(loss, s["params"])
    # the gradients as one vector, as a program that reduces them over ranks in one call has them
    return {"logits": logits.detach(), "loss": loss.detach(), "grads": torch.cat([x.reshape(-1) for x in grads])}


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------

def _op_flops(n_tok, D, T=64):
    """The operator per (batch, head, token) in the chunked form: forward, backward."""
    return n_tok * (10 * T * D + 6 * D * D), n_tok * (22 * T * D + 12 * D * D + 4 * T * T)


def work(case):
    kind, B = case["kind"], case["B"]
    if kind in ("decode", "prefill", "forward", "grad"):
        H, D = case["H"], case["D"]
    if kind == "decode":
        eb = 2 if case["dtype"] == "bf16" else 4
        return {"bytes": B * H * (2 * D * D + 7 * D) * eb, "flops": B * H * 6 * D * D}
    if kind in ("prefill", "forward"):
        n, eb = B * H * case["L"], 2 if case["dtype"] == "bf16" else 4
        states = 2 if case.get("h0") else 1
        return {"bytes": n * D * (6 * eb + 4) + states * B * H * D * D * 4, "flops": _op_flops(n, D)[0]}
    if kind == "grad":
        n = B * H * case["L"]
        # q..g and dO read, o and six gradients written; h_final and its cotangent, h0 and its gradient
        return {"bytes": n * D * 14 * 4 + (4 if case["h0"] else 2) * B * H * D * D * 4, "flops": sum(_op_flops(n, D))}
    n, c = B * case["L"], e2e_lm.LMConfig()
    d, p, m = c.d_model, c.proj_dim, c.mlp_mult * c.d_model
    mat = d * (6 * p + c.n_heads) + p * d + 3 * d * m       # one block's matrix entries
    op = sum(_op_flops(n * c.n_heads, c.d_head))
    block_flops = 6 * n * mat + op
    if kind == "block":
        return {"bytes": 4 * (4 * n * d + 3 * mat), "flops": block_flops}
    layers, V = c.n_layers, c.vocab_size
    return {"bytes": 4 * (n * V + 3 * (layers * mat + V * d)), "flops": layers * block_flops + 6 * n * d * V}


# ---------------------------------------------------------------------------------------------
# how far a correct implementation may be off
# ---------------------------------------------------------------------------------------------

def tolerance(case):
    # about four times the distance from the 64-bit result (fp32 operator 3e-7 .. 5e-7, bf16x3
    # products 7e-6, a layer 2e-6 .. 4e-6, the whole model 6e-6)
    kind = case["kind"]
    if kind == "decode":
        return {"rel": 1e-2, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 2e-6, "max": 4e-5}
    if kind == "prefill":
        # a bf16 state is rounded after every token of the tail
        return {"rel": 1e-2, "max": 0.1} if case["state"] == "bf16" else {"rel": 2e-6, "max": 4e-5}
    if kind == "forward":
        return {"rel": 2e-6, "max": 4e-5}
    if kind == "grad":
        return {"rel": 3e-6, "max": 1e-4} if case["cfg"] == "highest" else {"rel": 4e-5, "max": 2e-3}
    if kind == "block":
        return {"rel": 2e-5, "max": 1e-3}
    return {"rel": 4e-5, "max": 4e-3}


# ---------------------------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------------------------

def _tokens64(q, k, v, w, b, g, scale, h, keep, state_round=None):
    """Token recurrence of (B, H, L, D) inputs; keep (B, L): False where a row starts from zero."""
    outs = []
    for t in range(q.shape[2]):
        h = torch.where(keep[:, t, None, None, None], h, torch.zeros_like(h))
        h = h * torch.exp(g[:, :, t].clamp(max=0.0))[..., None]
        erase = ((b[:, :, t] * k[:, :, t]).unsqueeze(-2) @ h).squeeze(-2)
        h = h + k[:, :, t][..., None] * (w[:, :, t] * v[:, :, t] - erase).unsqueeze(-2)
        outs.append((scale * q[:, :, t].unsqueeze(-2) @ h).squeeze(-2))
        if state_round is not None and t >= state_round[0]:
            h = h.to(state_round[1]).to(torch.float64)
    return torch.stack(outs, dim=2), h


def _chunks64(q, k, v, w, b, g, scale, h, bt=64, eps=0.0):
    """Chunked form of the recurrence, the in-chunk coupling damped by 1 - eps; differentiable."""
    B, H, L, D = q.shape
    cut = lambda x: x.reshape(B, H, L // bt, bt, D)  # noqa: E731
    q, k, v, w, b, g = map(cut, (q, k, v, w, b, g))
    gc = g.cumsum(-2)
    mid = 0.5 * gc[..., -1:, :]
    up, down = torch.exp(gc - mid), torch.exp(mid - gc)
    kd = (k * down).transpose(-1, -2).contiguous()
    strict = torch.ones(bt, bt, dtype=q.dtype, device=q.device).tril(-1)
    akk = ((b * k * up) @ kd) * strict
    aqk = scale * ((q * up) @ kd) * (strict + torch.eye(bt, dtype=q.dtype, device=q.device))
    eye = torch.eye(bt, dtype=q.dtype, device=q.device).expand_as(akk)
    inv = torch.linalg.solve_triangular(eye + (1.0 - eps) * akk, eye, upper=False, unitriangular=True)
    eg = torch.exp(gc)
    wx, u = inv @ (b * k * eg), inv @ (w * v)
    qg, gl = scale * q * eg, gc[..., -1, :]
    kg = (k * torch.exp(gl[..., None, :] - gc)).transpose(-1, -2).contiguous()
    outs = []
    for c in range(L // bt):
        vn = u[:, :, c] - wx[:, :, c] @ h
        outs.append(qg[:, :, c] @ h + aqk[:, :, c] @ vn)
        h = torch.exp(gl[:, :, c])[..., None] * h + kg[:, :, c] @ vn
    return torch.stack(outs, dim=2).reshape(B, H, L, D), h


def _block64(p, x, c):
    B, L, _ = x.shape
    H, D = c.n_heads, c.d_head

    def conv(name, y):
        wt = p[name + ".weight"]
        K = wt.shape[1]
        out = p[name + ".bias"] + y * wt[:, K - 1]
        for s in range(1, K):
            out = out + F.pad(y[:, :-s], (0, 0, s, 0)) * wt[:, K - 1 - s]
        return out

    heads = lambda y: y.reshape(B, L, H, D)  # noqa: E731
    rms = lambda y, sc: y * torch.rsqrt(y.pow(2).mean(-1, keepdim=True) + 1e-6) * sc  # noqa: E731
    q, k, v = (heads(F.silu(conv(n + "_conv", x @ p[n + "_proj.weight"]))) for n in "qkv")
    v = v.clamp(-50.0, 50.0)
    q, k = (y * torch.rsqrt((y * y).sum(-1, keepdim=True) + 1e-6) for y in (q, k))
    b, w = (heads(torch.sigmoid(x @ p[n + ".weight"] + p[n + ".bias"])) for n in ("erase_gate", "write_gate"))
    ld = -torch.exp(p["decay_a"].clamp(-20, 20)) * F.softplus(x @ p["decay_proj.weight"] + p["decay_proj.bias"])
    g = (-ld.abs().clamp(max=c.g_max)).unsqueeze(-1).expand(B, L, H, D)
    o, _ = _chunks64(*(y.transpose(1, 2) for y in (q, k, v, w, b, g)), D ** -0.5,
                     torch.zeros(B, H, D, D, dtype=x.dtype, device=x.device))
    o = o.transpose(1, 2).reshape(B, L, H * D)
    x = x + (rms(o, p["mixer_out_norm.scale"]) * F.silu(x @ p["out_gate.weight"])) @ p["out_proj.weight"]
    h2 = rms(x, p["mlp_norm.scale"])
    return x + (F.silu(h2 @ p["gate_proj.weight"]) * (h2 @ p["up_proj.weight"])) @ p["down_proj.weight"]


def _params64(module):
    return {n: p.detach().double().requires_grad_(True) for n, p in module.named_parameters()}


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    f64 = lambda t: t.detach().double()  # noqa: E731
    if kind in ("decode", "prefill"):
        B, H, D = case["B"], case["H"], case["D"]
        xs = [f64(x) for x in s["xs"]]
        if kind == "prefill":
            ids, L = s["ids"], case["L"]
            keep = torch.cat([torch.ones(B, 1, dtype=torch.bool, device=DEV), ids[:, 1:] == ids[:, :-1]], dim=1)
            rnd = (L // 64 * 64, torch.bfloat16) if case["state"] == "bf16" else None
            o, h = _tokens64(*xs, s["scale"], torch.zeros(B, H, D, D, dtype=torch.float64, device=DEV), keep, rnd)
            return {"o": o, "h": h}
        q, k, v, w, b, g = xs
        if case["fuse"]:
            q, k = (x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
            b, w = torch.sigmoid(b), torch.sigmoid(w)
            g = -torch.exp(f64(s["a_log"]))[:, None] * F.softplus(g + f64(s["dt_bias"]))
        keep = torch.ones(B, 1, dtype=torch.bool, device=DEV) if s["reset"] is None else (s["reset"] <= 0)[:, None]
        one = lambda x: x.unsqueeze(2)  # noqa: E731
        o, h = _tokens64(*map(one, (q, k, v, w, b, g)), s["scale"], f64(s["state"]), keep)
        if s["tau"] is not None:
            nrm = h.square().sum(dim=(-2, -1), keepdim=True).sqrt().clamp(min=1e-12)
            h = h * (s["tau"] / nrm).clamp(max=1.0)
        return {"o": o[:, :, 0], "state": h}
    if kind in ("forward", "grad"):
        B, H, D = case["B"], case["H"], case["D"]
        prod = case.get("cfg") == "prod"
        grad = kind == "grad"
        xs = [f64(x).requires_grad_(grad) for x in s["xs"]]
        h0 = torch.zeros(B, H, D, D, dtype=torch.float64, device=DEV) if s["h0"] is None else f64(s["h0"])
        h0.requires_grad_(grad)
        with torch.set_grad_enabled(grad):
            o, h = _chunks64(*xs, s["scale"], h0, bt=128 if prod else 64, eps=1e-3 if prod else 0.0)
        if not grad:
            return {"o": o, "h": h}
        leaves = xs + ([h0] if s["h0"] is not None else [])
        grads = torch.autograd.grad((o, h), leaves, (f64(s["do"]), f64(s["dh"])))
        return {"o": o.detach(), "h": h.detach(), "grads": list(grads)}
    cfg = e2e_lm.LMConfig()
    if kind == "block":
        p, x = _params64(s["block"]), f64(s["x"]).requires_grad_(True)
        y = _block64(p, x, cfg)
        return {"y": y.detach(), "grads": list(torch.autograd.grad(y, [x] + list(p.values()), f64(s["dy"])))}
    p = _params64(s["model"])
    ids = s["ids"]
    x = p["embed"][ids]
    for i in range(cfg.n_layers):
        pre = f"blocks.{i}."
        x = _block64({n[len(pre):]: t for n, t in p.items() if n.startswith(pre)}, x, cfg)
    x = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * p["final_norm.scale"]
    logits = x @ p["embed"].t()
    V = logits.shape[-1]
    loss = F.cross_entropy(logits[:, :-1].reshape(-1, V), ids[:, 1:].reshape(-1))
    grads = torch.autograd.grad(loss, list(p.values()))
    return {"logits": logits.detach(), "loss": loss.detach(), "grads": torch.cat([t.reshape(-1) for t in grads])}
