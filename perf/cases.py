"""The work a user of this framework has it do, as cases that can be timed and compared.

A case is a dict of plain values.  ``listed()`` gives the ones that are quoted, ``draw``
more of the same ranges; ``prepare`` makes what a program holds before the call,
``run`` is one pass through the public entry points, ``exact`` the same values in
float64 from plain torch.  Kinds:

  scan         mamba3_siso_hip, the prefill operator
  carry        mamba3_siso_hip_carry, a prefill that continues a recurrent carry
  grads        mamba3_siso_hip under autograd: the training pair, all eleven gradients
  decode       rnn_step_hip, one token for a batch, in place on the carry
  layer        Mamba3Layer.forward
  layer_train  Mamba3Layer.train_forward and its backward
  generate     Mamba3Stack.step_graph, one token for a batch through the whole backbone
  stack_train  Mamba3Stack.loss_and_grads, a whole training step

The rotation angle of a carry is a point on the circle, and values on either side of
its wrap are the same angle, so it is not among the outputs compared: the rope'd key
of the same carry, which is, holds it.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sigma-0_amd"))

import mamba3_rocm as m3  # noqa: E402
from mamba3_rocm import layer as m3_layer, stack as m3_stack  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
VOCAB = 2112          # the LOB models' message vocabulary, as the backbone benchmark has it
# The gradient of dt_bias in a bf16 layer is a sum of cancelling sequence sums: its
# distance from float64 grows with the length (1% at 1024 tokens, 4% at 1500-3000, 40%
# at 12288 for a random cotangent), so longer training cases could not be compared.
_LAYER_TRAIN_L = 2048
NAMES = ("Q", "K", "V", "ADT", "DT", "Trap", "Q_bias", "K_bias", "Angles", "D", "Z")


def listed():
    return [
        # the reference benchmark's smallest configuration: two short sequences in float32
        dict(name="scan_f32_small", kind="scan", io="f32", B=2, L=1024, H=8, Hqk=8, N=64, P=64, R=16, chunk=64),
        # one prompt of odd length for a conversation that goes on: latency is what counts
        dict(name="prompt_carry_bf16", kind="carry", io="bf16", B=1, L=613, H=24, Hqk=24, N=128, P=64, R=32, chunk=64),
        # the headline prefill: a batch of sequences in bf16
        dict(name="scan_bf16_batch", kind="scan", io="bf16", B=8, L=4096, H=32, Hqk=32, N=128, P=64, R=32, chunk=64),
        # one long context: few (batch, head) pairs, many chunks
        dict(name="scan_bf16_long", kind="scan", io="bf16", B=1, L=32768, H=32, Hqk=32, N=128, P=64, R=32, chunk=128),
        # the same batch in float32, which is what the model itself hands its scan
        dict(name="scan_f32_batch", kind="scan", io="f32", B=8, L=4096, H=32, Hqk=32, N=128, P=64, R=32, chunk=64),
        # training through the operator in bf16
        dict(name="grads_bf16_batch", kind="grads", io="bf16", B=8, L=4096, H=32, Hqk=32, N=128, P=64, R=32, chunk=64),
        # and in float32, with a ragged length
        dict(name="grads_f32_ragged", kind="grads", io="f32", B=4, L=2999, H=32, Hqk=32, N=128, P=64, R=32, chunk=64),
        # one generated token for a full serving batch at the operator
        dict(name="decode_batch", kind="decode", io="bf16", B=512, H=32, N=128, P=64, R=32),
        # a mixer layer at the width and length its per-layer times are published for
        dict(name="layer_bf16_13000", kind="layer", io="bf16", B=1, L=13000, d_model=1024),
        # a mixer layer's training step with as many tokens as the backbone benchmark's batch:
        # the largest case (the lengths of the training cases: see _LAYER_TRAIN_L)
        dict(name="layer_train_bf16", kind="layer_train", io="bf16", B=32, L=1531, d_model=768),
        # generation: a serving batch through the twelve-layer backbone, one token each
        dict(name="generate_64", kind="generate", io="bf16", B=64, layers=12, d_model=768),
        # a small training step of whole blocks and the head, ragged length
        dict(name="stack_train_small", kind="stack_train", io="bf16", B=4, L=1501, layers=2, d_model=768),
    ]


def _log_int(rng, lo, hi):
    """Log-uniform over [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["scan", "scan", "scan", "carry", "grads", "grads", "decode", "layer", "layer_train", "generate",
                       "stack_train"])
    io = rng.choice(["bf16", "f32"])
    if kind in ("scan", "carry", "grads"):
        # the model's geometry mostly (rope_fraction 0.5, sometimes 1.0), else smaller ones
        N, P, R = rng.choice([(128, 64, 32)] * 4 + [(128, 64, 64), (64, 64, 16), (64, 32, 16)])
        H = rng.choice([4, 8, 16, 24, 32])
        Hqk = H if rng.random() < 0.8 else rng.choice([1, H // 2])
        B = _log_int(rng, 1, 16)
        most = (1 << 20) // (B * H)               # token-heads of the largest listed scan
        if kind == "grads":
            most = (most * 2) // (5 if io == "f32" else 3)
        L = _log_int(rng, 65 if kind != "grads" else 200, min(32768, most))
        return dict(kind=kind, io=io, B=B, L=L, H=H, Hqk=Hqk, N=N, P=P, R=R, chunk=rng.choice([64, 64, 64, 128]))
    if kind == "decode":
        return dict(kind=kind, io=io, B=_log_int(rng, 1, 512), H=rng.choice([8, 16, 24, 32]),
                    **rng.choice([dict(N=128, P=64, R=32), dict(N=128, P=64, R=64), dict(N=64, P=64, R=16)]))
    d_model = rng.choice([256, 512, 768, 1024])
    if kind == "generate":
        return dict(kind=kind, io="bf16", B=_log_int(rng, 1, 512), layers=rng.choice([4, 8, 12]), d_model=d_model)
    B = _log_int(rng, 1, 8 if kind == "layer" else 24)
    most = 49152 * 768 // (d_model * B)
    if kind == "stack_train":
        return dict(kind=kind, io="bf16", B=B, L=_log_int(rng, 100, min(_LAYER_TRAIN_L, most // 4)),
                    layers=rng.choice([1, 2, 3]), d_model=d_model)
    return dict(kind=kind, io="bf16", B=B, L=_log_int(rng, 100, min(16384 if kind == "layer" else _LAYER_TRAIN_L, most)),
                d_model=d_model)


# ------------------------------------------------------------------ inputs


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * scale


def _uniform(g, lo, hi, *shape):
    return torch.rand(*shape, generator=g, device="cuda") * (hi - lo) + lo


def _carry_inputs(g, B, H, N, P, R):
    """A recurrent carry in the middle of a sequence: theta, ssm, k, v."""
    return (_uniform(g, 0.0, 2.0 * math.pi, B, H, R), _randn(g, B, H, P, N, scale=0.1),
            _randn(g, B, H, N, scale=N ** -0.5), _randn(g, B, H, P))


def _scan_inputs(c, seed):
    """The benchmark configurations' distributions: x, z ~ N(0, 1); dt = softplus(N(-2,
    0.5)); A = -exp(U[log 1, log 16]) per head; B, C and the biases ~ N(0, 1) / sqrt(N);
    angle rates ~ U[-pi, pi]; trapezoid logits ~ U(0, 1)."""
    g, dt = _gen(seed), DTYPES[c["io"]]
    B, L, H, N, P, R = (c[k] for k in ("B", "L", "H", "N", "P", "R"))
    d = dict(Q=_randn(g, B, L, c["Hqk"], N, scale=N ** -0.5).to(dt), K=_randn(g, B, L, c["Hqk"], N, scale=N ** -0.5).to(dt),
             V=_randn(g, B, L, H, P).to(dt), Z=_randn(g, B, L, H, P).to(dt))
    DT = torch.nn.functional.softplus(_randn(g, B, H, L, scale=0.5) - 2.0)
    A = -torch.exp(_uniform(g, 0.0, math.log(16.0), H))
    d.update(DT=DT, ADT=A[None, :, None] * DT, Trap=_uniform(g, 0.0, 1.0, B, H, L),
             Angles=_uniform(g, -math.pi, math.pi, B, L, H, R), Q_bias=_randn(g, H, N, scale=N ** -0.5),
             K_bias=_randn(g, H, N, scale=N ** -0.5), D=_randn(g, H))
    return g, tuple(d[k] for k in NAMES)


def _decode_inputs(c, seed):
    g, dt = _gen(seed), DTYPES[c["io"]]
    B, H, N, P, R = (c[k] for k in ("B", "H", "N", "P", "R"))
    carry = _carry_inputs(g, B, H, N, P, R)
    dts = torch.nn.functional.softplus(_randn(g, B, H, scale=0.5) - 2.0)
    A = -torch.exp(_uniform(g, 0.0, math.log(16.0), H))
    t = (_randn(g, B, H, P).to(dt), _randn(g, B, H, P).to(dt), _randn(g, B, H, N, scale=N ** -0.5).to(dt),
         _randn(g, B, H, N, scale=N ** -0.5).to(dt), A * dts, dts, torch.sigmoid(_uniform(g, 0.0, 1.0, B, H)),
         _uniform(g, -math.pi, math.pi, B, H, R))
    return carry, t, _randn(g, H, N, scale=N ** -0.5), _randn(g, H, N, scale=N ** -0.5), _randn(g, H)


def _layer_inputs(c, seed):
    p = m3_layer.init_params(c["d_model"], seed, "cuda")
    g = _gen(seed + 1)
    x = _randn(g, c["B"], c["L"], c["d_model"]).to(DTYPES[c["io"]])
    return p, x, _randn(g, c["B"], c["L"], c["d_model"]).to(DTYPES[c["io"]])


def _stack_inputs(c, seed):
    p = m3_stack.init_params(VOCAB, c["d_model"], c["layers"], seed, "cuda")
    g = _gen(seed + 1)
    if c["kind"] == "generate":
        H = 2 * c["d_model"] // 64
        ids = torch.randint(VOCAB, (c["B"],), generator=g, device="cuda")
        return p, ids, [_carry_inputs(g, c["B"], H, 128, 64, 32) for _ in range(c["layers"])]
    ids = torch.randint(VOCAB, (c["B"], c["L"] + 1), generator=g, device="cuda")
    return p, ids[:, :-1].contiguous(), ids[:, 1:].contiguous()


def prepare(case, seed):
    c, kind = case, case["kind"]
    s = dict(kind=kind, chunk=c.get("chunk", 64))
    if kind in ("scan", "carry", "grads"):
        g, s["args"] = _scan_inputs(c, seed)
        if kind == "carry":
            s["init"] = _carry_inputs(g, c["B"], c["H"], c["N"], c["P"], c["R"])
        if kind == "grads":
            s["dout"] = _randn(g, c["B"], c["L"], c["H"], c["P"]).to(DTYPES[c["io"]])
            for t in s["args"]:
                t.requires_grad_(True)
    elif kind == "decode":
        s["carry"], s["t"], s["bb"], s["cb"], s["D"] = _decode_inputs(c, seed)
    elif kind in ("layer", "layer_train"):
        p, s["x"], dout = _layer_inputs(c, seed)
        if kind == "layer_train":
            s["dout"] = dout
            s["x"].requires_grad_(True)
            for t in p.values():
                t.requires_grad_(True)
        s["layer"] = m3.Mamba3Layer(p, c["d_model"], dtype=DTYPES[c["io"]])
    elif kind == "generate":
        p, s["ids"], s["state"] = _stack_inputs(c, seed)
        s["step"] = m3.Mamba3Stack(p, c["d_model"], dtype=DTYPES[c["io"]]).step_graph(s["state"])
    else:
        p, s["ids"], s["targets"] = _stack_inputs(c, seed)
        s["stack"] = m3.Mamba3Stack(p, c["d_model"], dtype=DTYPES[c["io"]])
    return s


def run(s):
    kind = s["kind"]
    if kind == "scan":
        return m3.mamba3_siso_hip(*s["args"], chunk_size=s["chunk"])
    if kind == "carry":
        out, (_, ssm, k, v) = m3.mamba3_siso_hip_carry(*s["args"], chunk_size=s["chunk"], initial_carry=s["init"])
        return out, ssm, k, v
    if kind == "grads":
        out = m3.mamba3_siso_hip(*s["args"], chunk_size=s["chunk"])
        return (out.detach(), *torch.autograd.grad(out, s["args"], s["dout"]))
    if kind == "decode":
        (_, ssm, k, v), y = m3.rnn_step_hip(s["carry"], s["t"], s["bb"], s["cb"], s["D"])
        return y, ssm, k, v
    if kind == "layer":
        return s["layer"].forward(s["x"])
    if kind == "layer_train":
        layer = s["layer"]
        out = layer.train_forward(s["x"])
        return (out.detach(), *torch.autograd.grad(out, [s["x"], *(layer.params[k] for k in m3_layer.PARAM_NAMES)],
                                                   s["dout"]))
    if kind == "generate":
        logp = s["step"](s["ids"])
        return (logp, *(t for _, ssm, k, v in s["state"] for t in (ssm, k, v)))
    loss, grads = s["stack"].loss_and_grads(s["ids"], s["targets"])
    return loss, grads


# ------------------------------------------------------------------ what a pass cannot do without


def _scan_work(B, L, H, Hqk, N, P, R, es):
    """(bytes, flops) of a forward scan: every input read and the output written once;
    the contractions at 64-token chunks."""
    return (B * L * (2 * Hqk * N * es + H * (3 * P * es + 12 + 4 * R)), B * L * H * (128.0 * N + 128.0 * P + 4.0 * P * N))


def _layer_work(B, L, d, es):
    """(bytes, flops) of one mixer layer: x in, out, the two projections and the scan."""
    di, H = 2 * d, 2 * d // 64
    dp = 2 * di + 256 + 3 * H + 32
    scan = _scan_work(B, L, H, 1, 128, 64, 32, es)[1]
    return B * L * 2 * d * es + (d * dp + di * d) * es, scan + 2.0 * B * L * (d * dp + di * d)


def work(case):
    c, kind = case, case["kind"]
    es = 2 if c["io"] == "bf16" else 4
    if kind in ("scan", "carry", "grads"):
        B, L, H, Hqk, N, P, R = (c[k] for k in ("B", "L", "H", "Hqk", "N", "P", "R"))
        by, fl = _scan_work(B, L, H, Hqk, N, P, R, es)
        if kind == "carry":
            by += 8 * B * H * (P * N + N + P + R)
        if kind == "grads":                       # forward, then inputs and dOut in, gradients out
            by, fl = 3 * by, 3 * fl
        return dict(bytes=by, flops=fl)
    if kind == "decode":
        B, H, N, P, R = (c[k] for k in ("B", "H", "N", "P", "R"))
        return dict(bytes=B * H * (8 * (P * N + R + N + P) + (2 * P + 2 * N) * es + 12 + 4 * R + 4 * P),
                    flops=8.0 * B * H * P * N)
    if kind in ("layer", "layer_train"):
        by, fl = _layer_work(c["B"], c["L"], c["d_model"], es)
        return dict(bytes=by, flops=fl) if kind == "layer" else dict(bytes=3 * by, flops=3 * fl)
    d, n, B = c["d_model"], c["layers"], c["B"]
    H = 2 * d // 64
    weights = d * (4 * d + 288 + 3 * H) + 2 * d * d + d * d           # the mixer's two and the gate's Dense
    if kind == "generate":
        return dict(bytes=n * (weights * es + B * H * 8 * (64 * 128 + 32 + 128 + 64)) + VOCAB * d * 4 + B * VOCAB * 4,
                    flops=2.0 * B * (n * weights + VOCAB * d) + 8.0 * n * B * H * 64 * 128)
    by, fl = _layer_work(B, c["L"], d, es)
    rows = B * c["L"]
    return dict(bytes=3 * n * (by + d * d * es) + 12 * rows * VOCAB,
                flops=3 * (n * (fl + 2.0 * rows * d * d) + 2.0 * rows * d * VOCAB))


def tolerance(case):
    """About four times the distance between correct computations at the same precision.
    bf16 holds 8 bits, so outputs differ by 2e-3 or so and gradients, which pass several
    bf16 operands and are summed over whole sequences, by up to 7e-3; a layer and a
    backbone round between their parts too.  float32 sums in another order differ by
    1e-6, the sequence sums of the angle and decay gradients by 1e-5."""
    kind, bf = case["kind"], case["io"] == "bf16"
    if kind in ("scan", "carry"):
        return {"rel": 0.01} if bf else {"rel": 1e-5, "max": 1e-3}
    if kind == "grads":
        return {"rel": 0.03, "max": 0.9} if bf else {"rel": 5e-5, "max": 1e-2}
    if kind == "decode":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "layer":
        return {"rel": 0.015}
    if kind == "generate":
        return {"rel": 0.03, "max": 0.9}
    return {"rel": 0.03, "max": 0.9}


# ------------------------------------------------------------------ the same values in float64


def _rope(x, th):
    """Interleaved pairs (2j, 2j + 1), j < R, of x (B, L, H, N) turned by th (B, L, H, R)."""
    R = th.shape[-1]
    if R == 0:
        return x
    cs, sn = torch.cos(th), torch.sin(th)
    x0, x1 = x[..., 0:2 * R:2], x[..., 1:2 * R:2]
    turned = torch.stack([x0 * cs - x1 * sn, x0 * sn + x1 * cs], -1).flatten(-2)
    return torch.cat([turned, x[..., 2 * R:]], -1)


def _scan64(Q, K, V, ADT, DT, Trap, Q_bias, K_bias, Angles, D, Z, init=None):
    """The operator in float64: 64-token chunks, the state carried from chunk to chunk.
    Returns (y, (ssm, k, v)) with the carry after the last token."""
    B, L, Hqk, N = Q.shape
    H, P = V.shape[2:]
    C = 64
    head = torch.arange(H, device=V.device) // (H // Hqk)
    th = torch.cumsum(torch.tanh(Angles) * math.pi * DT.transpose(1, 2)[..., None], 1)
    sig = torch.sigmoid(Trap)
    gamma = DT * sig
    nxt = torch.nn.functional.pad((DT * (1.0 - sig))[..., 1:], (0, 1))
    if init is not None:
        th = th + init[0][:, None]
    q, k = Q[:, :, head] + Q_bias, K[:, :, head] + K_bias
    skip = (q * k).sum(-1) * gamma.transpose(1, 2) + D
    q, k = _rope(q, th), _rope(k, th)
    last_k = k[:, -1]
    k = k * (gamma + nxt).transpose(1, 2)[..., None]
    nc = -(-L // C)

    def chunks(t):                                   # (B, L, H, .) -> (B, H, nc, C, .)
        t = torch.nn.functional.pad(t, (0, 0, 0, 0, 0, nc * C - L))
        return t.reshape(B, nc, C, H, -1).permute(0, 3, 1, 2, 4).contiguous()
    qc, kc, vc = chunks(q), chunks(k), chunks(V)
    A = torch.cumsum(torch.nn.functional.pad(ADT, (0, nc * C - L)).reshape(B, H, nc, C), -1)
    below = torch.ones(C, C, dtype=torch.bool, device=V.device).tril(-1)
    decay = torch.exp((A[..., :, None] - A[..., None, :]).masked_fill(~below, -math.inf))
    y = ((qc @ kc.transpose(-1, -2).contiguous()) * decay) @ vc
    kw = (kc * torch.exp(A[..., -1:] - A)[..., None]).transpose(-1, -2).contiguous()
    qw, end = qc * torch.exp(A)[..., None], torch.exp(A[..., -1])
    if init is None:
        h = torch.zeros(B, H, N, P, dtype=V.dtype, device=V.device)
    else:                                            # the trapezoid's term with the token before
        h = init[1].transpose(-1, -2) + (DT * (1.0 - sig))[..., 0, None, None] * init[2][..., :, None] * init[3][..., None, :]
    off = []
    for i in range(nc):
        off.append(qw[:, :, i] @ h)
        h = end[:, :, i, None, None] * h + kw[:, :, i] @ vc[:, :, i]
    y = (y + torch.stack(off, 2)).permute(0, 2, 3, 1, 4).reshape(B, nc * C, H, P)[:, :L]
    y = y + skip[..., None] * V
    return y * torch.nn.functional.silu(Z), (h.transpose(-1, -2), last_k, V[:, -1])


def _step64(carry, t, bb, cb, D):
    """One token of the recurrence in float64: (y, (ssm, k, v))."""
    theta, h, kp, vp = carry
    x, z, Bt, Ct, adt, dt, trap, ang = t
    th = (theta + torch.tanh(ang) * math.pi * dt[..., None])[:, None]
    b, c = _rope((Bt + bb)[:, None], th)[:, 0], _rope((Ct + cb)[:, None], th)[:, 0]
    e, w = torch.exp(adt)[..., None, None], dt[..., None, None]
    tr = trap[..., None, None]
    h = e * (h + (1.0 - tr) * w * vp[..., :, None] * kp[..., None, :]) + tr * w * x[..., :, None] * b[..., None, :]
    y = (h * c[..., None, :]).sum(-1) + D[:, None] * x
    return y * torch.nn.functional.silu(z), (h, b, x)


def _rms(x, scale):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * scale


def _mixer64(p, x, carry=None):
    """The mixer layer in float64 on x (B, L, d); with a carry, one token (L = 1)."""
    B, L, _ = x.shape
    H, N, di = p["D"].shape[0], p["B_norm"].shape[0], p["out_norm"].shape[0]
    proj = x @ p["in_proj"]
    z, xv, b, cc, dd, da, trap, ang = torch.split(proj, [di, di, N, N, H, H, H, proj.shape[-1] - 2 * di - 2 * N - 3 * H], -1)
    b, cc = _rms(b, p["B_norm"]), _rms(cc, p["C_norm"])
    A = torch.clamp(-torch.nn.functional.softplus(da), max=-1e-4)
    dt = torch.nn.functional.softplus(dd + p["dt_bias"])
    heads = lambda t: t.reshape(B, L, H, di // H)  # noqa: E731
    ang = ang[:, :, None].expand(B, L, H, ang.shape[-1])
    if carry is None:
        rows = lambda t: t.transpose(1, 2)  # noqa: E731
        y, new = _scan64(cc[:, :, None], b[:, :, None], heads(xv), rows(A * dt), rows(dt), rows(trap), p["C_bias"],
                         p["B_bias"], ang, p["D"], heads(z))
    else:
        one = lambda t: t[:, 0]  # noqa: E731
        wide = lambda t: t.expand(B, H, N)  # noqa: E731
        y, new = _step64(carry, (one(heads(xv)), one(heads(z)), wide(b), wide(cc), one(A * dt), one(dt),
                                 torch.sigmoid(one(trap)), one(ang)), p["B_bias"], p["C_bias"], p["D"])
    return _rms(y.reshape(B, L, di), p["out_norm"]) @ p["out_proj"], new


def _block64(lp, x, carry=None):
    """A prenorm half_glu1 block in float64."""
    xn = torch.nn.functional.layer_norm(x, x.shape[-1:], lp["ln_scale"], lp["ln_bias"], 1e-6)
    y, new = _mixer64(lp["mixer"], xn, carry)
    g = torch.nn.functional.gelu(y, approximate="tanh")
    return x + g * torch.sigmoid(g @ lp["out2_w"] + lp["out2_b"]), new


def _to64(v):
    if isinstance(v, dict):
        return {k: _to64(x) for k, x in v.items()}
    if isinstance(v, (list, tuple)):
        return [_to64(x) for x in v]
    return v.detach().double()


def _leaves(v):
    if isinstance(v, dict):
        return [t for x in v.values() for t in _leaves(x)]
    if isinstance(v, list):
        return [t for x in v for t in _leaves(x)]
    return [v]


def _filled(v, grads):
    if isinstance(v, dict):
        return {k: _filled(x, grads) for k, x in v.items()}
    if isinstance(v, list):
        return [_filled(x, grads) for x in v]
    g = next(grads)
    return torch.zeros_like(v) if g is None else g


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("scan", "carry"):
        g, args = _scan_inputs(c, seed)
        if kind == "scan":
            return _scan64(*_to64(args))[0]
        init = _to64(_carry_inputs(g, c["B"], c["H"], c["N"], c["P"], c["R"]))
        y, (ssm, k, v) = _scan64(*_to64(args), init=init)
        return y, ssm, k, v
    if kind == "grads":
        g, args = _scan_inputs(c, seed)
        dout = _randn(g, c["B"], c["L"], c["H"], c["P"]).to(DTYPES[c["io"]]).double()
        args = [t.requires_grad_(True) for t in _to64(args)]
        y = _scan64(*args)[0]
        return (y.detach(), *torch.autograd.grad(y, args, dout))
    if kind == "decode":
        y, (ssm, k, v) = _step64(*(_to64(x) for x in _decode_inputs(c, seed)))
        return y, ssm, k, v
    if kind in ("layer", "layer_train"):
        p, x, dout = (_to64(v) for v in _layer_inputs(c, seed))
        if kind == "layer":
            return _mixer64(p, x)[0]
        leaves = [x.requires_grad_(True), *(p[k].requires_grad_(True) for k in m3_layer.PARAM_NAMES)]
        y = _mixer64(p, x)[0]
        return (y.detach(), *torch.autograd.grad(y, leaves, dout))
    p, ids, more = _stack_inputs(c, seed)
    p = _to64(p)
    if kind == "generate":
        x, news = p["embed"][ids][:, None], []
        for lp, carry in zip(p["layers"], more):
            x, new = _block64(lp, x, _to64(carry))
            news += new
        return (torch.log_softmax(x[:, 0] @ p["decoder_w"] + p["decoder_b"], -1), *news)
    leaves = [t.requires_grad_(True) for t in _leaves(p)]
    x = p["embed"][ids]
    for lp in p["layers"]:
        x = _block64(lp, x)[0]
    logp = torch.log_softmax(x @ p["decoder_w"] + p["decoder_b"], -1)
    loss = -logp.gather(-1, more[..., None]).mean()
    grads = torch.autograd.grad(loss, leaves, allow_unused=True)
    return loss.detach(), _filled(p, iter(grads))
