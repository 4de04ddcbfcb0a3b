"""The calls whose time counts: the fused ops as a training or inference program makes them.

Every case goes through the public functions of ``nuvla_forge_amd.kernels``,
eagerly, forward and (with ``train``) backward through autograd:

  seam      ``fused_adaln_residual_rmsnorm`` on [b * t, n] rows
  swiglu    ``fused_swiglu`` on [m, h]
  ce        ``chunked_cross_entropy`` on hidden [m, d], lm_head [v, d], the
            default chunk_size
  gate_up   ``fused_gate_up_swiglu`` on x [m, d], weights [h, d]

``dtype`` is the program's precision: ``bf16`` (every tensor bf16), ``fp32``,
or ``amp`` (fp32 parameters and residual stream under bf16 autocast, branch
outputs and conditioning in bf16).
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from nuvla_forge_amd.kernels import (
    chunked_cross_entropy,
    fused_adaln_residual_rmsnorm,
    fused_gate_up_swiglu,
    fused_swiglu,
)

DEVICE = "cuda"
IGNORE = -100


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    def seam(name, b, t, n, dtype):
        return dict(name=name, op="seam", b=b, t=t, n=n, dtype=dtype, train=True)

    def swiglu(name, m, h, dtype):
        return dict(name=name, op="swiglu", m=m, h=h, dtype=dtype, train=True)

    def ce(name, m, d, v, dtype, ignored):
        return dict(name=name, op="ce", m=m, d=d, v=v, dtype=dtype, ignored=ignored, train=True)

    def gate_up(name, m, d, h, dtype):
        return dict(name=name, op="gate_up", m=m, d=d, h=h, dtype=dtype, train=True)

    return [
        # the trajectory planner's DiT block at its training batch of 8: 6
        # waypoints of width 384 under autocast, where latency counts
        seam("seam_planner", 8, 6, 384, "amp"),
        # the same block over a large batch of scenes: many samples of few tokens
        seam("seam_planner_batch", 2048, 6, 384, "amp"),
        # a DiT of image-sized token grids, the headline shape
        seam("seam_base", 8, 1024, 1024, "bf16"),
        # the largest: a long-sequence DiT beyond the caches
        seam("seam_large", 32, 2048, 2048, "bf16"),
        # the vision encoder's MLP: 8 samples x 6 views x 196 patches, 384 -> 1536
        swiglu("swiglu_encoder", 9408, 1536, "bf16"),
        # a language-model MLP over 65536 tokens, beyond the caches
        swiglu("swiglu_large", 65536, 5632, "bf16"),
        # the reasoning head in training: 8 x 64 text tokens, fp32 lm_head
        # under autocast, every seventh token masked
        ce("ce_head", 512, 384, 32000, "amp", 1 / 7),
        # a 2048-wide language model's head, 10 % of the tokens masked
        ce("ce_lm", 4096, 2048, 32000, "bf16", 0.1),
        # a narrow head over many tokens and an odd vocabulary: several chunks
        ce("ce_tall_odd", 12289, 384, 50001, "bf16", 0.03),
        # the reasoning head trained in full precision
        ce("ce_fp32", 512, 384, 32000, "fp32", 1 / 7),
        # the vision encoder's gate/up projections in training (fp32
        # parameters under autocast)
        gate_up("gate_up_encoder", 9408, 384, 1536, "amp"),
        # a 2048-wide language model's gate/up projections
        gate_up("gate_up_wide", 4096, 2048, 5632, "bf16"),
    ]


def _log_int(rng, lo, hi, step=1):
    x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(x / step)) * step))


def draw(rng):
    op = rng.choice(["seam", "seam", "swiglu", "ce", "ce", "gate_up"])
    train = rng.random() < 0.8  # else inference: the forward alone
    if op == "seam":
        n = _log_int(rng, 256, 4096, 8)
        t = _log_int(rng, 1, 2048)
        dtype = rng.choice(["amp", "amp", "bf16", "bf16", "fp32"])
        most = (1 << 27 if dtype == "bf16" else 1 << 26) // n
        rows = _log_int(rng, 48, min(65536, most))
        return dict(op=op, b=max(1, rows // t), t=min(t, rows), n=n, dtype=dtype, train=train)
    if op == "swiglu":
        h = _log_int(rng, 256, 5632)
        return dict(op=op, m=_log_int(rng, 48, 65536), h=h,
                    dtype=rng.choice(["bf16", "bf16", "bf16", "fp32"]) if h < 2816 else "bf16",
                    train=train)
    if op == "ce":
        dtype = rng.choice(["amp", "bf16", "bf16", "fp32"])
        d = _log_int(rng, 256, 2048, 8)
        v = _log_int(rng, 1000, 128256)
        most = (1e11 if dtype == "fp32" else 1.4e12) / (6.0 * d * v)  # no dearer than ce_lm
        return dict(op=op, m=_log_int(rng, 48, int(max(49, min(16384, most)))), d=d, v=v,
                    dtype=dtype, ignored=round(rng.uniform(0.0, 0.5), 3), train=True)
    d = _log_int(rng, 256, 2048, 8)
    h = _log_int(rng, 512, 5632, 8)
    most = 5.6e11 / (12.0 * d * h)
    return dict(op=op, m=_log_int(rng, 48, int(min(65536, most))), d=d, h=h,
                dtype=rng.choice(["amp", "bf16"]), train=train)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _types(case):
    """(residual / parameter type, branch / conditioning type)"""
    return {"bf16": (torch.bfloat16, torch.bfloat16), "fp32": (torch.float32, torch.float32),
            "amp": (torch.float32, torch.bfloat16)}[case["dtype"]]


def _kept(case):
    """Rows of a ce case that count."""
    return case["m"] - int(case["m"] * case["ignored"])


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    wide, narrow = _types(case)

    def rand(*shape, std=1.0, mean=0.0, dtype=wide):
        return torch.empty(shape, device=DEVICE).normal_(mean, std, generator=g).to(dtype)

    s = {"case": case}
    if case["op"] == "seam":
        b, t, n = case["b"], case["t"], case["n"]
        # the block's conditioning: one [B, 6 N] projection, used as chunk(6) views
        cond = rand(b, 6 * n, std=0.1, dtype=narrow).chunk(6, dim=-1)
        s["leaves"] = [rand(b * t, n), rand(b * t, n, dtype=narrow), cond[2],
                       rand(n, std=0.02, mean=1.0), cond[1], cond[0]]
        s["up"] = [rand(b * t, n), rand(b * t, n)]
    elif case["op"] == "swiglu":
        m, h = case["m"], case["h"]
        s["leaves"] = [rand(m, h), rand(m, h)]
        s["up"] = [rand(m, h)]
    elif case["op"] == "ce":
        m, d, v = case["m"], case["d"], case["v"]
        s["leaves"] = [rand(m, d), rand(v, d, std=0.02)]
        targets = torch.randint(0, v, (m,), device=DEVICE, generator=g)
        masked = torch.rand(m, device=DEVICE, generator=g).argsort()[: m - _kept(case)]
        targets[masked] = IGNORE
        s["targets"] = targets
    else:
        m, d, h = case["m"], case["d"], case["h"]
        s["leaves"] = [rand(m, d), rand(h, d, std=d ** -0.5), rand(h, d, std=d ** -0.5)]
        s["up"] = [rand(m, h, dtype=narrow)]
    for x in s["leaves"]:
        x.requires_grad_(case["train"])
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _forward(s):
    case, leaves = s["case"], s["leaves"]
    if case["op"] == "seam":
        return fused_adaln_residual_rmsnorm(*leaves, tokens_per_sample=case["t"])
    if case["op"] == "swiglu":
        return (fused_swiglu(*leaves),)
    if case["op"] == "ce":
        return (chunked_cross_entropy(*leaves, s["targets"], ignore_index=IGNORE),)
    return (fused_gate_up_swiglu(*leaves),)


def run(s):
    case = s["case"]
    with torch.autocast(DEVICE, dtype=torch.bfloat16, enabled=case["dtype"] == "amp"):
        if not case["train"]:
            with torch.no_grad():
                return list(_forward(s))
        outs = _forward(s)
    return [*outs, *torch.autograd.grad(outs, s["leaves"], s.get("up"))]


# ---------------------------------------------------------------------------
# what a pass cannot do without, and what it may be off by
# ---------------------------------------------------------------------------
def work(case):
    w, n = (torch.finfo(t).bits // 8 for t in _types(case))
    train = case["train"]
    if case["op"] == "seam":
        rows, small = case["b"] * case["t"] * case["n"], case["b"] * case["n"]
        forward = rows * (w + n + 2 * w) + 3 * small * n + case["n"] * w
        # the backward's own reads and writes (x, y and the conditioning again: they are
        # inputs of another call by then)
        backward = rows * (w + n + 2 * w + w + n) + small * 5 * n + 2 * case["n"] * w
        return {"bytes": forward + backward * train, "flops": 0}
    if case["op"] == "swiglu":
        return {"bytes": (3 + 5 * train) * case["m"] * case["h"] * w, "flops": 0}
    if case["op"] == "ce":
        m, d, v = case["m"], case["d"], case["v"]
        return {"bytes": 2 * w * (m * d + v * d) + 8 * m, "flops": 6.0 * _kept(case) * d * v}
    m, d, h = case["m"], case["d"], case["h"]
    forward = w * (m * d + 2 * h * d) + n * m * h
    backward = n * m * h + w * (m * d + 2 * h * d)
    return {"bytes": forward + backward * train, "flops": 4.0 * (1 + 2 * train) * m * d * h}


def tolerance(case):
    # 16-bit results: the rounding of each, of the operands of the products
    # and of what is kept between the calls is 2^-9 at most, about 2e-3 in the norm
    # (4e-3 through two products); fp32: sums in another order
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    return {"rel": 1.6e-2}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _exact_forward(s, x):
    case = s["case"]
    if case["op"] == "seam":
        b, t, n = case["b"], case["t"], case["n"]
        res, y, gate, weight, scale, shift = x
        h = res.view(b, t, n) + gate.unsqueeze(1) * y.view(b, t, n)
        xhat = h * torch.rsqrt(h.square().mean(-1, keepdim=True) + 1e-6)
        out = xhat * weight * (1 + scale.unsqueeze(1)) + shift.unsqueeze(1)
        return h.view(b * t, n), out.view(b * t, n)
    if case["op"] == "swiglu":
        return (F.silu(x[0]) * x[1],)
    if case["op"] == "ce":
        return (F.cross_entropy(x[0] @ x[1].T, s["targets"], ignore_index=IGNORE),)
    return (F.silu(x[0] @ x[1].T) * (x[0] @ x[2].T),)


def exact(case, seed):
    s = prepare(case, seed)
    train = case["train"]
    x = [v.detach().double().requires_grad_(train) for v in s["leaves"]]
    outs = _exact_forward(s, x)
    if not train:
        return list(outs)
    up = [u.double() for u in s["up"]] if "up" in s else None
    return [*(o.detach() for o in outs), *torch.autograd.grad(outs, x, up)]
