"""The work that users of this library have it do, as timed cases.

Every case goes through the public Python entry points: the trainable and
forward-only GDN2 and Mamba2 operators, the two prologues and the output
epilogue.  ``listed()`` gives the named cases, ``draw(rng)`` further ones of
the same ranges, ``prepare`` / ``run`` one pass, ``work`` what the pass cannot
do without, ``exact`` the same results from plain torch in 64 bits and
``tolerance`` how far another correct implementation may be from them.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "atomic_ai_hybrid-v0.1_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

_DT = {"bf16": torch.bfloat16, "fp32": torch.float32}
_ES = {"bf16": 2, "fp32": 4}


def listed():
    return [
        # a serving loop that extends each sequence by one block of tokens: the
        # smallest call, with the state of the tokens before it
        dict(name="gdn2_extend", op="gdn2_fwd", B=1, T=64, H=8, K=128, dtype="bf16", h0=True),
        # the float32 forward of the validation configuration
        dict(name="gdn2_fwd_fp32", op="gdn2_fwd", B=1, T=512, H=4, K=64, dtype="fp32", h0=False),
        # prefill of one long document
        dict(name="gdn2_prefill_long", op="gdn2_fwd", B=1, T=32768, H=16, K=128, dtype="bf16", h0=False),
        # a training step of the model's GDN2 layer (d_model 768, six heads)
        dict(name="gdn2_train_model", op="gdn2_train", B=8, T=4096, H=6, K=128, dtype="bf16", h0=False),
        # a training step of the benchmark's GDN2 layer
        dict(name="gdn2_train_large", op="gdn2_train", B=4, T=8192, H=16, K=128, dtype="bf16", h0=False),
        # scoring / prefill with the Mamba2 layer of the forward configuration
        dict(name="mamba2_fwd", op="mamba2_fwd", B=2, T=4096, H=32, P=64, N=128, chunk=128, dtype="bf16", h0=False),
        # a training step of the model's Mamba2 layer (d_inner 1536 over eight heads, chunks of 256)
        dict(name="mamba2_train_model", op="mamba2_train", B=8, T=4096, H=8, P=192, N=128, chunk=256, dtype="bf16",
             h0=False),
        # a training step of the benchmark's Mamba2 layer
        dict(name="mamba2_train_large", op="mamba2_train", B=4, T=8192, H=16, P=128, N=128, chunk=128, dtype="bf16",
             h0=False),
        # a float32 training step, as for checking a recipe before going to bf16
        dict(name="mamba2_train_fp32", op="mamba2_train", B=2, T=2048, H=8, P=64, N=64, chunk=64, dtype="fp32",
             h0=False),
        # the GDN2 layer's input side in training: convolutions, normalisation and gates
        dict(name="gdn2_prologue", op="gdn2_prologue", B=4, T=4096, H=16, D=128),
        # the Mamba2 layer's input side in training: dt / B / C projections and the convolution
        dict(name="mamba2_proj", op="mamba2_proj", B=8, T=4096, H=8, D=192, N=128),
        # the Mamba2 layer's output side in training: norm and gate
        dict(name="out_norm_gate", op="norm_gate", variant="mamba2", B=8, T=4096, H=8, D=192),
    ]


def _log_int(rng, lo, hi):
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    op = rng.choice(["gdn2_fwd", "gdn2_train", "mamba2_fwd", "mamba2_train", "gdn2_prologue", "mamba2_proj",
                     "norm_gate"])
    while True:
        if op in ("gdn2_fwd", "gdn2_train"):
            c = dict(op=op, B=_log_int(rng, 1, 8), T=64 * _log_int(rng, 1, 512), H=_log_int(rng, 1, 24),
                     K=rng.choice([64, 128, 128]), dtype=rng.choice(["bf16", "bf16", "bf16", "fp32"]),
                     h0=rng.random() < 0.5)
            n, most = c["B"] * c["T"] * c["H"] * c["K"], 1 << 26 if c["dtype"] == "bf16" else 1 << 22
        elif op in ("mamba2_fwd", "mamba2_train"):
            chunk = rng.choice([64, 128, 256])
            P = rng.choice([64, 128, 192])
            c = dict(op=op, B=_log_int(rng, 1, 8), T=chunk * _log_int(rng, 1, 32768 // chunk), H=_log_int(rng, 1, 64),
                     P=P, N=128 if P == 192 else rng.choice([64, 128]), chunk=chunk,
                     dtype=rng.choice(["bf16", "bf16", "bf16", "fp32"]), h0=rng.random() < 0.5)
            n, most = c["B"] * c["T"] * c["H"] * P, 1 << 26 if c["dtype"] == "bf16" else 1 << 21
        elif op == "gdn2_prologue":
            D = rng.choice([64, 128])
            c = dict(op=op, B=_log_int(rng, 1, 8), T=128 * _log_int(rng, 1, 128), H=512 * rng.randint(1, 4) // D, D=D)
            n, most = c["B"] * c["T"] * c["H"] * D, 1 << 25
        elif op == "mamba2_proj":
            D = rng.choice([64, 128])
            c = dict(op=op, B=_log_int(rng, 1, 8), T=128 * _log_int(rng, 1, 128), H=512 * rng.randint(1, 4) // D, D=D,
                     N=rng.choice([64, 128]))
            d = c["H"] * D
            n, most = c["B"] * c["T"] * d * (d + 2 * c["N"]), 8 * 4096 * 1536 * 1792
        else:
            D = rng.choice([64, 128])
            c = dict(op=op, variant=rng.choice(["gdn2", "mamba2"]), B=_log_int(rng, 1, 8), T=_log_int(rng, 1, 16384),
                     H=512 * rng.choice([1, 2, 3, 4, 6, 8]) // D, D=D)
            n, most = c["B"] * c["T"] * c["H"] * D, 1 << 26
        if n <= most:
            return c


# ------------------------------------------------------------------ inputs
def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)


def _core_inputs(c, gen):
    """GDN2: q, k normalised, v, the gates and the log decay; Mamba2: dt, x, B,
    C and A, in the distributions of the benchmark configurations."""
    dt = _DT[c["dtype"]]
    if c["op"].startswith("gdn2"):
        shp = (c["B"], c["T"], c["H"], c["K"])
        q, k = (torch.nn.functional.normalize(_randn(gen, *shp), dim=-1) for _ in range(2))
        v = _randn(gen, *shp)
        w, b = (torch.sigmoid(_randn(gen, *shp)) for _ in range(2))
        g = torch.nn.functional.logsigmoid(3.0 + _randn(gen, *shp))
        x = [t.to(dt) for t in (q, k, v, w, b)] + [g]
        h0 = _randn(gen, c["B"], c["H"], c["K"], c["K"]) if c["h0"] else None
        up = shp
    else:
        shp, bt = (c["B"], c["T"], c["H"], c["P"]), (c["B"], c["T"], c["N"])
        step = torch.nn.functional.softplus(-2.0 + 0.5 * _randn(gen, *shp))
        xx = _randn(gen, *shp)
        Bm, Cm = (_randn(gen, *bt) / math.sqrt(c["N"]) for _ in range(2))
        A = -torch.exp(math.log(16.0) * torch.rand(c["H"], generator=gen, device="cuda"))
        x = [t.to(dt) for t in (step, xx, Bm, Cm)] + [A]
        h0 = _randn(gen, c["B"], c["H"], c["P"], c["N"]) if c["h0"] else None
        up = shp
    # the operators return float32, so the gradient that comes back is float32
    do = _randn(gen, *up) if c["op"].endswith("_train") else None
    if c["op"] == "mamba2_train":
        # half the squared distance of y to a target: the gradient is y - target.  (A gradient
        # that has nothing to do with y leaves dA a sum that cancels to 1e-4 of its terms.)
        h = torch.zeros(c["B"], c["H"], c["P"], c["N"], dtype=torch.float64, device="cuda")
        y, _ = _mamba2_64(*(t.double() for t in x), h if h0 is None else h0.double())
        do = y.float() - do
    return x, h0, do


def _side_inputs(c, gen):
    """What the layer's projections hand to the prologues and the epilogue, the
    parameters (float32) and the cotangents of every output."""
    bf = torch.bfloat16
    shp, d = (c["B"], c["T"], c["H"], c["D"]), c["H"] * c["D"]
    row = shp[:2] + (d,)
    if c["op"] == "gdn2_prologue":
        q, k, v, b, w = (_randn(gen, *row).to(bf) for _ in range(5))
        f = (_randn(gen, *row) - 3.0).to(bf)
        x = [q, k, v, 0.5 * _randn(gen, 3, d, 4), 0.1 * _randn(gen, 3, d), b, w, f, 0.1 * _randn(gen, c["H"])]
        cots = [_randn(gen, *shp).to(bf) for _ in range(5)] + [_randn(gen, *shp)]
    elif c["op"] == "mamba2_proj":
        n = c["N"]
        x = [_randn(gen, c["B"], c["T"], 2 * d).to(bf), 0.5 * _randn(gen, d, 4), 0.1 * _randn(gen, d),
             0.5 / math.sqrt(d) * _randn(gen, d, d), torch.full((d,), -2.0, device="cuda"),
             _randn(gen, d, n) / math.sqrt(d * n), _randn(gen, d, n) / math.sqrt(d * n),
             math.log(16.0) * torch.rand(c["H"], generator=gen, device="cuda")]
        cots = [_randn(gen, *shp).to(bf) for _ in range(2)] + [_randn(gen, *shp[:2], n).to(bf) for _ in range(2)]
        cots += [_randn(gen, c["H"])]
    else:
        y = _randn(gen, *shp)
        if c["variant"] == "mamba2":   # the gate is the second half of the in_proj output
            gate = _randn(gen, c["B"], c["T"], 2 * d).to(bf)[..., d:]
        else:
            gate = _randn(gen, *row).to(bf)
        x = [y, gate, 1.0 + 0.1 * _randn(gen, d)]
        cots = [_randn(gen, *row).to(bf)]
    return x, cots


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    st = dict(case=case)
    if case["op"].startswith(("gdn2_p", "mamba2_p", "norm")):
        st["x"], st["cots"] = _side_inputs(case, gen)
        train = True
    else:
        st["x"], st["h0"], st["do"] = _core_inputs(case, gen)
        train = st["do"] is not None
    if train:
        st["x"] = [t.detach().requires_grad_(True) for t in st["x"]]
    return st


def run(st):
    c, x = st["case"], st["x"]
    op = c["op"]
    if op in ("gdn2_fwd", "gdn2_train"):
        from atomic_ops import kernel_trainable_B6 as G
        if op == "gdn2_fwd":
            return G.gdn2_pallas_forward(*x, 1.0, st["h0"])
        out = G.gdn2_pallas_forward_trainable(*x, 1.0, st["h0"])
        return out + torch.autograd.grad(out[0], x, st["do"])
    if op in ("mamba2_fwd", "mamba2_train"):
        from atomic_ops import kernel_mamba2_trainable_B6 as M
        if op == "mamba2_fwd":
            return M.mamba2_pallas_forward(*x, c["chunk"], st["h0"])
        out = M.mamba2_pallas_forward_trainable_B6(*x, c["chunk"], st["h0"])
        return out + torch.autograd.grad(out[0], x, st["do"])
    if op == "gdn2_prologue":
        from atomic_ops.prologue import GDN2Prologue
        out = GDN2Prologue.apply(*x, c["H"])
    elif op == "mamba2_proj":
        from atomic_ops.prologue import Mamba2ProjPrologue
        out = Mamba2ProjPrologue.apply(*x, c["H"])
    else:
        from atomic_ops import norm_gate
        f = norm_gate.mamba2_out_norm_gate if c["variant"] == "mamba2" else norm_gate.gdn2_out_norm_gate
        out = (f(*x),)
    return tuple(out) + torch.autograd.grad(out, x, st["cots"])


# ------------------------------------------------------------------ work and tolerance
def work(case):
    """Each input read once, each output written once; the products of the
    chunked forms (64-row GDN2 chunks, the case's Mamba2 chunk)."""
    c, op = case, case["op"]
    rows = c["B"] * c["T"]
    if op.startswith("gdn2_") and op != "gdn2_prologue":
        es, K, C = _ES[c["dtype"]], c["K"], 64
        n, st = rows * c["H"] * K, c["B"] * c["H"] * K * K
        by = n * (5 * es + 4) + n * 4 + st * 4 * (2 if c["h0"] else 1)
        fl = rows * c["H"] / C * (10 * C * C * K + 6 * C * K * K + C ** 3 / 3)
        if op == "gdn2_train":
            by += n * 4 + n * (5 * es + 4)
            fl += rows * c["H"] / C * (20 * C * C * K + 12 * C * K * K + 4 * C ** 3)
        return dict(bytes=by, flops=fl)
    if op in ("mamba2_fwd", "mamba2_train"):
        es, P, N, C = _ES[c["dtype"]], c["P"], c["N"], c["chunk"]
        n, bn, st = rows * c["H"] * P, rows * N, c["B"] * c["H"] * P * N
        by = (2 * n + 2 * bn) * es + n * 4 + st * 4 * (2 if c["h0"] else 1)
        fl = rows * (2 * C * N + c["H"] * (2 * C * P + 4 * P * N))
        if op == "mamba2_train":
            by += n * 4 + (2 * n + 2 * bn) * es
            fl += rows * (4 * C * N + c["H"] * (6 * C * P + 8 * P * N))
        return dict(bytes=by, flops=fl)
    d = c["H"] * c["D"]
    n = rows * d
    if op == "gdn2_prologue":
        # six projections in, five bf16 outputs and g; their cotangents in, six gradients out
        return dict(bytes=n * (12 + 14 + 14 + 12), flops=n * 200)
    if op == "mamba2_proj":
        w = d + 2 * c["N"]
        # x_bc in; x, dt, B, C out and their cotangents in; the whole in_proj gradient out; weights in and out
        return dict(bytes=rows * (2 * d + 4 * (2 * d + 2 * c["N"]) + 4 * d) + 8 * d * w, flops=6.0 * rows * d * w)
    # y, gate, dout in; out, dy, dgate out
    return dict(bytes=n * (4 + 2 + 2 + 2 + 4 + 2), flops=n * 60)


def tolerance(case):
    """About four times the distance between what the library gave for these
    ranges and the 64-bit results: float32 1e-6, bf16 GDN2 6e-3 (its gradients
    of b and g), bf16 Mamba2 1e-2 (its gradient of dt), the others 4e-3."""
    if case.get("dtype") == "fp32":
        return {"rel": 1e-5}
    if case["op"] in ("mamba2_fwd", "mamba2_train"):
        return {"rel": 3e-2}
    return {"rel": 2.4e-2 if case["op"] in ("gdn2_fwd", "gdn2_train") else 1.6e-2}


# ------------------------------------------------------------------ 64-bit results
def _unit_lower_inverse(a):
    """(I + a)^-1 of strictly lower triangular a: the product of I + (-a)^(2^i)."""
    p = -a
    eye = torch.eye(a.shape[-1], dtype=a.dtype, device=a.device)
    inv, n = eye + p, 2
    while n < a.shape[-1]:
        p = p @ p
        inv = inv + inv @ p
        n *= 2
    return inv


def _gdn2_64(q, k, v, w, b, g, h):
    B, T, H, K = q.shape
    C = 64
    q, k, v, w, b, g = (t.reshape(B, T // C, C, H, K).permute(0, 3, 1, 2, 4).contiguous() for t in (q, k, v, w, b, g))
    gc = g.cumsum(3)
    e, last = gc.exp(), gc[..., -1:, :]
    kt = (k * (-gc).exp()).transpose(-1, -2).contiguous()
    qg, kb = q * e, b * k * e
    inv = _unit_lower_inverse((kb @ kt).tril(-1))
    wp, u, aqk = inv @ kb, inv @ (w * v), (qg @ kt).tril()
    kg = (k * (last - gc).exp()).transpose(-1, -2).contiguous()
    decay = last.exp().transpose(-1, -2)
    out = []
    for n in range(T // C):
        vn = u[:, :, n] - wp[:, :, n] @ h
        out.append(qg[:, :, n] @ h + aqk[:, :, n] @ vn)
        h = h * decay[:, :, n] + kg[:, :, n] @ vn
    return torch.stack(out, 2).permute(0, 2, 3, 1, 4).reshape(B, T, H, K), h


def _mamba2_64(dt, x, Bm, Cm, A, h):
    B, T, H, P = dt.shape
    N, C = Bm.shape[-1], 64
    nt = T // C
    cum = (dt * A[:, None]).reshape(B, nt, C, H * P).cumsum(2)
    dbx = (dt * x).reshape(B, nt, C, H * P)
    Bc, Cc = Bm.reshape(B, nt, C, N), Cm.reshape(B, nt, C, N)
    cb = (Cc @ Bc.transpose(-1, -2).contiguous()).tril()
    e, last = cum.exp(), cum[:, :, -1:]
    y = e * (cb @ (dbx * (-cum).exp()))
    add = Bc.transpose(-1, -2).contiguous() @ (dbx * (last - cum).exp())   # [B, nt, N, H P]
    end = last.exp()
    h = h.reshape(B, H * P, N).transpose(1, 2)
    off = []
    for n in range(nt):
        off.append(Cc[:, n] @ h)
        h = h * end[:, n] + add[:, n]
    y = y + e * torch.stack(off, 1)
    return y.reshape(B, T, H, P), h.transpose(1, 2).reshape(B, H, P, N)


def _conv_silu(u, w, bias):
    """Causal depthwise convolution over [B, T, d] and SiLU."""
    T, taps = u.shape[1], w.shape[1]
    up = torch.nn.functional.pad(u, (0, 0, taps - 1, 0))
    z = sum(up[:, j:j + T] * w[:, j] for j in range(taps)) + bias
    return z * torch.sigmoid(z)


def _gdn2_prologue_64(x, H):
    q, k, v, cw, cb, b, w, f, a = x
    shp = q.shape[:2] + (H, -1)
    q, k, v = (_conv_silu(u, cw[i], cb[i]).reshape(shp) for i, u in enumerate((q, k, v)))
    q, k = (t * torch.rsqrt((t * t).sum(-1, keepdim=True) + 1e-12) for t in (q, k))
    v = v.clamp(-50.0, 50.0)
    g = -a.exp()[:, None] * torch.nn.functional.softplus(f.reshape(shp))
    return q, k, v, torch.sigmoid(w).reshape(shp), torch.sigmoid(b).reshape(shp), g


def _mamba2_proj_64(x, H):
    u, cw, cb, w_dt, b_dt, w_b, w_c, a_log = x
    u = u[..., :w_dt.shape[0]]
    shp = u.shape[:2] + (H, -1)
    dt = torch.nn.functional.softplus(u @ w_dt + b_dt)
    dt = dt.clamp(float(torch.tensor(1e-2, dtype=torch.bfloat16)), 1.0)   # the step's bounds are bf16 values
    return _conv_silu(u, cw, cb).reshape(shp), dt.reshape(shp), u @ w_b, u @ w_c, -a_log.exp()


def _norm_gate_64(x, variant):
    y, gate, w = x
    y = y.reshape(gate.shape)
    n = y * torch.rsqrt((y * y).mean(-1, keepdim=True) + 1e-6) * w
    if variant == "gdn2":
        gate = gate.clamp(-1e2, 1e2)
    out = n * gate * torch.sigmoid(gate)
    return (out.clamp(-3e2, 3e2) if variant == "mamba2" else out,)


def exact(case, seed):
    c, st = case, prepare(case, seed)
    train = st["x"][0].requires_grad
    x = [t.detach().double().requires_grad_(train) for t in st["x"]]
    with torch.set_grad_enabled(train):
        if c["op"] in ("gdn2_fwd", "gdn2_train"):
            h = torch.zeros(c["B"], c["H"], c["K"], c["K"], dtype=torch.float64, device="cuda")
            out = _gdn2_64(*x, h if st["h0"] is None else st["h0"].double())
        elif c["op"] in ("mamba2_fwd", "mamba2_train"):
            h = torch.zeros(c["B"], c["H"], c["P"], c["N"], dtype=torch.float64, device="cuda")
            out = _mamba2_64(*x, h if st["h0"] is None else st["h0"].double())
        elif c["op"] == "gdn2_prologue":
            out = _gdn2_prologue_64(x, c["H"])
        elif c["op"] == "mamba2_proj":
            out = _mamba2_proj_64(x, c["H"])
        else:
            out = _norm_gate_64(x, c["variant"])
        if not train:
            return out
        if c["op"] in ("gdn2_train", "mamba2_train"):
            return out + torch.autograd.grad(out[0], x, st["do"].double())
        return out + torch.autograd.grad(out, x, [t.double() for t in st["cots"]])
