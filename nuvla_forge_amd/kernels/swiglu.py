"""Fused SwiGLU on MI355X: ``out = silu(a) * b`` in one HBM pass.

Drop-in for ``nuvla_forge/kernels/swiglu.py``: the same ``_FusedSwiGLU``
autograd Function (``forward(ctx, a, b)``, ``backward`` returning ``(da, db)``,
swiglu.py:66-92) and the same ``fused_swiglu(a, b, force_reference=False)``
entry point (swiglu.py:95-106).  The forward and backward are the HIP kernels
``nf_swiglu_fwd`` / ``nf_swiglu_bwd``; the backward recomputes the sigmoid
from ``a`` instead of storing it.

Beyond the reference: ``fused_gate_up_swiglu`` moves the SwiGLU into the
epilogue of the gate/up projection GEMM (``nf_gemm_swiglu``), so a and b
never make the HBM round trip between the projections and the activation.
"""

from __future__ import annotations

import torch
import torch.nn.functional as F

from .. import _lib
from .reference import swiglu_ref
from .utils import check_devices, device_of, use_fused


def _check(a: torch.Tensor, b: torch.Tensor) -> None:
    if a.shape != b.shape:
        raise ValueError(f"fused_swiglu: shape mismatch {tuple(a.shape)} vs {tuple(b.shape)}")
    if a.dtype != b.dtype:
        raise TypeError(f"fused_swiglu: dtype mismatch {a.dtype} vs {b.dtype}")
    check_devices("fused_swiglu", "a", dict(a=a, b=b))
    _lib.dtype_code(a)


class _FusedSwiGLU(torch.autograd.Function):
    @staticmethod
    def forward(ctx, a, b):
        _check(a, b)
        a = a.contiguous()
        b = b.contiguous()
        out = torch.empty_like(a)
        L = _lib.lib()
        with device_of(a):
            _lib.check(
                L.nf_swiglu_fwd(a.data_ptr(), b.data_ptr(), out.data_ptr(), a.numel(),
                                _lib.dtype_code(a), _lib.stream_of(a)),
                "nf_swiglu_fwd",
            )
        ctx.save_for_backward(a, b)
        return out

    @staticmethod
    def backward(ctx, dout):
        a, b = ctx.saved_tensors
        check_devices("fused_swiglu backward", "a", dict(a=a, dout=dout))
        dout = dout.contiguous()
        if dout.dtype != a.dtype:
            dout = dout.to(a.dtype)
        da = torch.empty_like(a)
        db = torch.empty_like(b)
        L = _lib.lib()
        with device_of(a):
            _lib.check(
                L.nf_swiglu_bwd(dout.data_ptr(), a.data_ptr(), b.data_ptr(), da.data_ptr(),
                                db.data_ptr(), a.numel(), _lib.dtype_code(a), _lib.stream_of(a)),
                "nf_swiglu_bwd",
            )
        return da, db


class _FusedGateUpSwiGLU(torch.autograd.Function):
    """act = silu(x W_gate^T) * (x W_up^T) with the SwiGLU in the GEMM epilogue.

    forward: the inputs in bf16 (cast where they are not), then one
    ``nf_gemm_swiglu`` launch writes act and the bf16 a, b the backward needs.
    backward: ``nf_swiglu_bwd`` forms da, db from a, b and dact (sigmoid
    recomputed); ``nf_gemm_swiglu_bwd`` computes dx = da W_gate + db W_up,
    dW_gate = da^T x and dW_up = db^T x in one launch, each written once in
    its input's type (sums over K splits added in a fixed order).  Where
    ``nf_gemm_swiglu_bwd_wins`` says no (large all-bf16 products, sooner for dx
    alone), dx is two library GEMMs and both weight gradients come from
    ``nf_gemm_swiglu_wgrad``.
    """

    @staticmethod
    def forward(ctx, x, w_gate, w_up):
        check_devices("fused_gate_up_swiglu", "x", dict(x=x, w_gate=w_gate, w_up=w_up))
        ctx.dtypes = (x.dtype, w_gate.dtype, w_up.dtype)
        x, w_gate, w_up = _rows_bf16(x), _rows_bf16(w_gate), _rows_bf16(w_up)
        m, d = x.shape
        h = w_gate.shape[0]
        a = torch.empty((m, h), dtype=torch.bfloat16, device=x.device)
        b = torch.empty_like(a)
        act = torch.empty_like(a)
        L = _lib.lib()
        with device_of(x):
            _lib.check(
                L.nf_gemm_swiglu(x.data_ptr(), x.stride(0), w_gate.data_ptr(), w_gate.stride(0),
                                 w_up.data_ptr(), w_up.stride(0), a.data_ptr(), b.data_ptr(),
                                 act.data_ptr(), h, m, d, h, _lib.dtype_code(torch.bfloat16),
                                 _lib.stream_of(x)),
                "nf_gemm_swiglu",
            )
        ctx.save_for_backward(x, w_gate, w_up, a, b)
        return act

    @staticmethod
    def backward(ctx, dact):
        x, w_gate, w_up, a, b = ctx.saved_tensors
        check_devices("fused_gate_up_swiglu backward", "x", dict(x=x, dact=dact))
        dact = dact.to(torch.bfloat16).contiguous()
        da, db = torch.empty_like(a), torch.empty_like(b)
        L = _lib.lib()
        with device_of(a):
            _lib.check(
                L.nf_swiglu_bwd(dact.data_ptr(), a.data_ptr(), b.data_ptr(), da.data_ptr(),
                                db.data_ptr(), a.numel(), _lib.dtype_code(a), _lib.stream_of(a)),
                "nf_swiglu_bwd",
            )
        need = ctx.needs_input_grad
        m, d = x.shape
        h = a.shape[1]
        # the kernel writes fp32, bf16 or fp16: dx in x's type, both weight
        # gradients in one, theirs or fp32 where two are wanted and differ
        # (neither may round the other's gradient); any other type is cast to
        # from fp32
        need_x, need_g, need_u = need[:3]
        tx, tg, tu = ctx.dtypes
        cx = tx if tx in _lib.DTYPE_CODE else torch.float32
        cw = tg if need_g else tu
        if (need_g and need_u and tg != tu) or cw not in _lib.DTYPE_CODE:
            cw = torch.float32
        dx = torch.empty((m, d), dtype=cx, device=x.device) if need_x else None
        dwg = torch.empty((h, d), dtype=cw, device=x.device) if need_g else None
        dwu = torch.empty((h, d), dtype=cw, device=x.device) if need_u else None
        code = _lib.dtype_code(torch.bfloat16)
        one_x, one_w = need_x, need_g or need_u  # left to the one launch
        with device_of(x):
            st = _lib.stream_of(x)
            if (tx == tg == tu == torch.bfloat16
                    and not L.nf_gemm_swiglu_bwd_wins(m, d, h, one_w)):
                if one_x:
                    with torch.no_grad(), torch.autocast(x.device.type, enabled=False):
                        dx = torch.addmm(torch.mm(da, w_gate), db, w_up)
                    one_x = False
                if need_g and need_u:
                    nbytes = L.nf_gemm_swiglu_wgrad_workspace(m, d, h)
                    ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=x.device)
                    _lib.check(
                        L.nf_gemm_swiglu_wgrad(da.data_ptr(), db.data_ptr(), h, x.data_ptr(),
                                               x.stride(0), dwg.data_ptr(), dwu.data_ptr(), d,
                                               m, d, h, code, ws.data_ptr(), nbytes, st),
                        "nf_gemm_swiglu_wgrad",
                    )
                    one_w = False
            if one_x or one_w:
                if d % 8 == 0 and h % 8 == 0:  # other widths go to padded rows in the call
                    x, w_gate, w_up = (_vector_rows(t.detach()) for t in (x, w_gate, w_up))
                pg, pu = (_lib.ptr(dwg), _lib.ptr(dwu)) if one_w else (None, None)
                nbytes = L.nf_gemm_swiglu_bwd_workspace(m, d, h, one_x, bool(pg), bool(pu))
                ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=x.device)
                _lib.check(
                    L.nf_gemm_swiglu_bwd(da.data_ptr(), db.data_ptr(), h, x.data_ptr(),
                                         x.stride(0), w_gate.data_ptr(), w_gate.stride(0),
                                         w_up.data_ptr(), w_up.stride(0),
                                         dx.data_ptr() if one_x else None, _lib.dtype_code(cx),
                                         pg, pu, _lib.dtype_code(cw), m, d, h, code,
                                         ws.data_ptr(), nbytes, st),
                    "nf_gemm_swiglu_bwd",
                )
        return (dx.to(tx) if need_x else None, dwg.to(tg) if need_g else None,
                dwu.to(tu) if need_u else None)


def _gate_up_eager(x, w_gate, w_up):
    return F.silu(F.linear(x, w_gate)) * F.linear(x, w_up)


def fused_gate_up_swiglu(x: torch.Tensor, w_gate: torch.Tensor, w_up: torch.Tensor,
                         force_reference: bool = False) -> torch.Tensor:
    """``silu(x @ w_gate.T) * (x @ w_up.T)``: the gate/up half of a SwiGLU MLP
    (the reference's ``SwiGLUMLP``, model/dit.py:96-110) with the SwiGLU fused
    into the projection GEMM's epilogue.

    Args:
        x: [..., D] activations.
        w_gate, w_up: [H, D] projection weights (``nn.Linear.weight``); each
            may have its own row stride.
        force_reference: run the eager formulation (two Linears + silu * mul).

    The fused kernel computes in bf16 with fp32 accumulation: it runs when
    the inputs are bf16, or under bf16 autocast (as the Linears would); other
    dtypes take the two Linears and the fused SwiGLU kernel.  Host tensors
    take the eager formulation.  Gradients come back in each input's dtype.
    """
    if not use_fused(x, "fused_gate_up_swiglu", force_reference):
        return _gate_up_eager(x, w_gate, w_up)
    if w_gate.shape != w_up.shape or w_gate.dim() != 2 or x.shape[-1] != w_gate.shape[1]:
        raise ValueError(f"fused_gate_up_swiglu: x [..., D] and weights [H, D] expected, got "
                         f"{tuple(x.shape)}, {tuple(w_gate.shape)}, {tuple(w_up.shape)}")
    autocast_bf16 = (torch.is_autocast_enabled(x.device.type)
                     and torch.get_autocast_dtype(x.device.type) == torch.bfloat16)
    all_bf16 = x.dtype == w_gate.dtype == w_up.dtype == torch.bfloat16
    if not (all_bf16 or autocast_bf16):
        return fused_swiglu(F.linear(x, w_gate), F.linear(x, w_up))
    lead = x.shape[:-1]
    x2 = x.reshape(-1, x.shape[-1])
    # the plain call runs in C++; any other (None) takes the Function above
    act = _lib.native().gate_up(x2, w_gate, w_up)
    if act is None:
        with torch.autocast(x.device.type, enabled=False):
            act = _FusedGateUpSwiGLU.apply(x2, w_gate, w_up)
    return act.reshape(*lead, w_gate.shape[0])


def _rows_bf16(t: torch.Tensor) -> torch.Tensor:
    """bf16 with unit-stride rows (a cast / copy only when needed)."""
    t = t.to(torch.bfloat16)
    return t if t.stride(-1) == 1 else t.contiguous()


def _vector_rows(t: torch.Tensor) -> torch.Tensor:
    """``t`` with rows of whole 16-byte vectors (its width is a multiple of 8): a
    copy of a view whose base or row stride is not, which the backward would
    read element by element."""
    whole = t.data_ptr() % 16 == 0 and t.stride(0) % 8 == 0
    return t if whole else t.clone(memory_format=torch.contiguous_format)


def fused_swiglu(a: torch.Tensor, b: torch.Tensor, force_reference: bool = False) -> torch.Tensor:
    """SwiGLU: ``silu(a) * b``, fused into a single pass.

    Args:
        a: gate projection, any shape.
        b: up projection, same shape and dtype as ``a``.
        force_reference: run the eager PyTorch formulation instead.

    Host tensors take the eager formulation, as in the reference (swiglu.py:104).
    """
    if not use_fused(a, "fused_swiglu", force_reference):
        return swiglu_ref(a, b)
    # the plain call runs in C++; any other (None) takes the Function above
    out = _lib.native().swiglu(a, b)
    return out if out is not None else _FusedSwiGLU.apply(a, b)
