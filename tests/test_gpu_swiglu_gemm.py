"""SwiGLU fused into the gate/up projection GEMM (GPU).

``fused_gate_up_swiglu(x, w_gate, w_up)`` computes what the reference's
SwiGLUMLP computes before its down projection, ``silu(x W_gate^T) *
(x W_up^T)`` (model/dit.py:96-110), with one MFMA kernel whose epilogue
applies the activation.  Checked against the fp64 oracle on the same
bf16-rounded operands, forward and all three gradients, at 2e-2 norm-wise
relative error (the bf16 criterion), across tile-aligned, ragged (M, H not
multiples of the 256 x 128 tile), unaligned-D (register-copy loader) and
single-row shapes; against the eager composition; under bf16 autocast with
fp32 activations and weights; and fp32 inputs without autocast, which take
the two Linears and the fused SwiGLU kernel (1e-5).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from nuvla_forge_amd import _lib
from nuvla_forge_amd.kernels import fused_gate_up_swiglu
from oracle import numerics as on
from tests.helpers import gen, note, np64, randn

pytestmark = pytest.mark.gpu


def _oracle(x, wg, wu, dact):
    """fp64: a = x Wg^T, b = x Wu^T, act = silu(a) b and its gradients."""
    a, b = x @ wg.T, x @ wu.T
    act = on.swiglu_forward(a, b)
    da, db = on.swiglu_backward(a, b, dact)
    return act, da @ wg + db @ wu, da.T @ x, db.T @ x


def _inputs(m, d, h, dtype, dev, seed=0):
    g = gen(seed)
    x = randn((m, d), g, dtype, dev)
    wg = randn((h, d), g, dtype, dev, std=d ** -0.5)
    wu = randn((h, d), g, dtype, dev, std=d ** -0.5)
    dact = randn((m, h), g, dtype, dev)
    return x, wg, wu, dact


def _run(x, wg, wu, dact, **kw):
    leaves = [t.detach().requires_grad_(True) for t in (x, wg, wu)]
    act = fused_gate_up_swiglu(*leaves, **kw)
    act.backward(dact)
    torch.cuda.synchronize()
    return act.detach(), [t.grad for t in leaves]


@pytest.mark.parametrize("m,d,h", [(512, 384, 1536), (300, 200, 333), (64, 36, 100), (1, 8, 1),
                                   (2048, 1024, 2816)])
def test_gate_up_swiglu_matches_oracle(cuda, m, d, h):
    note(f"gemm swiglu m={m} d={d} h={h}")
    x, wg, wu, dact = _inputs(m, d, h, torch.bfloat16, cuda)
    act, (dx, dwg, dwu) = _run(x, wg, wu, dact)
    assert act.dtype == dx.dtype == dwg.dtype == torch.bfloat16
    ref = _oracle(np64(x), np64(wg), np64(wu), np64(dact))
    errs = {k: on.rel_err(np64(v), r)
            for k, v, r in zip(("act", "dx", "dwg", "dwu"), (act, dx, dwg, dwu), ref)}
    assert all(e <= 2e-2 for e in errs.values()), errs


# act alone takes the epilogue with 16-byte stores: tile edges (256 tokens, 128
# units), remainders of the 32-unit groups, output rows wider than H; beside it
# the same product with rows one element longer, which are not whole vectors
# and go out element by element, as a, b and act together do
@pytest.mark.parametrize("m,d,h,pad", [(256, 64, 128, 0), (257, 72, 136, 8), (255, 136, 24, 0),
                                       (31, 8, 8, 16), (513, 200, 264, 0), (1, 64, 1000, 8)])
@pytest.mark.parametrize("save", [True, False])
def test_gate_up_entry_rows_of_whole_vectors(cuda, m, d, h, pad, save):
    note(f"gate/up entry m={m} d={d} h={h} pad={pad} save={save}")
    x, wg, wu, _ = _inputs(m, d, h, torch.bfloat16, cuda, seed=m + h)
    L = _lib.lib()

    def run(ldo):
        outs = [torch.full((m, ldo), -7.0, dtype=torch.bfloat16, device=cuda)
                for _ in range(3 if save else 1)]
        ab = [o.data_ptr() for o in outs[1:]] if save else [None, None]
        _lib.check(L.nf_gemm_swiglu(x.data_ptr(), d, wg.data_ptr(), d, wu.data_ptr(), d, *ab,
                                    outs[0].data_ptr(), ldo, m, d, h,
                                    _lib.dtype_code(torch.bfloat16), _lib.stream_of(x)),
                   "nf_gemm_swiglu")
        torch.cuda.synchronize()
        for o in outs:
            assert (o[:, h:] == -7.0).all()  # nothing past a row's H
        return [np64(o[:, :h]) for o in outs]

    a, b = np64(x) @ np64(wg).T, np64(x) @ np64(wu).T
    want = [on.swiglu_forward(a, b), a, b]
    # each result is rounded to bf16 once: 2^-8 of it at most (8 significant
    # bits).  A sum of up to 200 products rounds ~13 times to 2^-24 of at most
    # sum |x w| ~ 10, 1e-5 absolute; silu(a) b carries that times |a|, |b| < 6.
    for got in (run(h + pad), run(h + pad + 1)):
        for g, w in zip(got, want):
            assert (np.abs(g - w) <= 2.0 ** -8 * np.abs(w) + 6e-5).all()


def test_gate_up_swiglu_weights_with_different_row_strides(cuda):
    """w_gate a column-slice view of a wider [H, 2D + 8] tensor (row stride
    2D + 8), w_up contiguous (row stride D): each weight is read through its
    own row stride."""
    note("gemm swiglu w_gate strided view, w_up contiguous")
    m, d, h = 300, 128, 384
    g = gen(7)
    x = randn((m, d), g, torch.bfloat16, cuda)
    wide = randn((h, 2 * d + 8), g, torch.bfloat16, cuda, std=d ** -0.5)
    wg = wide[:, 8:8 + d]
    wu = randn((h, d), g, torch.bfloat16, cuda, std=d ** -0.5)
    dact = randn((m, h), g, torch.bfloat16, cuda)
    assert wg.stride(0) == 2 * d + 8 and wu.stride(0) == d
    act, (dx, dwg, dwu) = _run(x, wg, wu, dact)
    ref = _oracle(np64(x), np64(wg), np64(wu), np64(dact))
    errs = {k: on.rel_err(np64(v), r)
            for k, v, r in zip(("act", "dx", "dwg", "dwu"), (act, dx, dwg, dwu), ref)}
    assert all(e <= 2e-2 for e in errs.values()), errs


def test_gate_up_swiglu_agrees_with_eager_composition(cuda):
    note("gemm swiglu vs eager composition")
    x, wg, wu, dact = _inputs(1024, 512, 1024, torch.bfloat16, cuda, seed=1)
    act, grads = _run(x, wg, wu, dact)
    act_e, grads_e = _run(x, wg, wu, dact, force_reference=True)
    assert on.rel_err(np64(act), np64(act_e)) < 1e-2
    for g, ge in zip(grads, grads_e):
        assert on.rel_err(np64(g), np64(ge)) < 2e-2


def test_gate_up_swiglu_under_autocast_keeps_input_dtypes(cuda):
    """fp32 activations and fp32 nn.Linear weights under bf16 autocast run
    the fused bf16 kernel; the gradients come back in fp32."""
    note("gemm swiglu autocast fp32 -> bf16")
    x, wg, wu, dact = _inputs(256, 384, 768, torch.float32, cuda, seed=2)
    leaves = [t.detach().requires_grad_(True) for t in (x, wg, wu)]
    with torch.autocast("cuda", dtype=torch.bfloat16):
        act = fused_gate_up_swiglu(*leaves)
    assert act.dtype == torch.bfloat16
    act.backward(dact.to(torch.bfloat16))
    torch.cuda.synchronize()
    assert all(t.grad.dtype == torch.float32 for t in leaves)
    xb, wgb, wub = (np64(t.to(torch.bfloat16)) for t in (x, wg, wu))
    ref = _oracle(xb, wgb, wub, np64(dact.to(torch.bfloat16)))
    got = [act] + [t.grad for t in leaves]
    assert all(on.rel_err(np64(v), r) <= 2e-2 for v, r in zip(got, ref))


def test_gate_up_swiglu_fp32_takes_the_composed_path(cuda):
    note("gemm swiglu fp32 without autocast")
    x, wg, wu, dact = _inputs(128, 64, 96, torch.float32, cuda, seed=3)
    act, (dx, dwg, dwu) = _run(x, wg, wu, dact)
    ref = _oracle(np64(x), np64(wg), np64(wu), np64(dact))
    for v, r in zip((act, dx, dwg, dwu), ref):
        assert on.rel_err(np64(v), r) <= 1e-5


def test_gate_up_swiglu_forward_is_deterministic_and_3d(cuda):
    note("gemm swiglu determinism, [B, T, D] input")
    x, wg, wu, _ = _inputs(4 * 96, 256, 640, torch.bfloat16, cuda, seed=4)
    x3 = x.view(4, 96, 256)
    a1 = fused_gate_up_swiglu(x3, wg, wu)
    a2 = fused_gate_up_swiglu(x3, wg, wu)
    assert a1.shape == (4, 96, 640) and torch.equal(a1, a2)
    ref = F.silu(x.float() @ wg.float().T) * (x.float() @ wu.float().T)
    assert on.rel_err(np64(a1.reshape(-1, 640)), np64(ref)) < 2e-2


def _wgrad(da, db, x, ldw=None):
    """Call nf_gemm_swiglu_wgrad on [M, H] views da, db and [M, D] view x."""
    from nuvla_forge_amd import _lib

    m, h = da.shape
    d = x.shape[1]
    ldw = ldw or d
    dwg_buf = torch.full((h, ldw), 7.0, dtype=torch.bfloat16, device=x.device)
    dwu_buf = torch.full_like(dwg_buf, 7.0)
    L = _lib.lib()
    nbytes = L.nf_gemm_swiglu_wgrad_workspace(m, d, h)
    ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=x.device)
    _lib.check(L.nf_gemm_swiglu_wgrad(da.data_ptr(), db.data_ptr(), da.stride(0), x.data_ptr(),
                                      x.stride(0), dwg_buf.data_ptr(), dwu_buf.data_ptr(), ldw,
                                      m, d, h, 1, ws.data_ptr(), nbytes, _lib.stream_of(x)),
               "nf_gemm_swiglu_wgrad")
    torch.cuda.synchronize()
    return dwg_buf, dwu_buf


# (M, D, H, row pad of da/db, row pad of x, row pad of dW): the headline DiT MLP
# (10 token slices), ragged H and D (the element-wise transpose), fewer tokens
# than one 8-token pad, and strided views with untouched pad columns.
@pytest.mark.parametrize("m,d,h,pab,px,pw", [
    (9408, 384, 1536, 0, 0, 0), (1000, 200, 333, 0, 0, 0), (5, 64, 96, 0, 0, 0),
    (777, 136, 264, 8, 16, 8), (3000, 1024, 2816, 0, 0, 0)])
def test_gate_up_wgrad_entry_matches_fp64(cuda, m, d, h, pab, px, pw):
    """dW_gate = da^T x, dW_up = db^T x from the same bf16 operands in fp64.
    The only rounding is fp32 accumulation and the final bf16 store, so the
    norm-wise error stays under 2^-8 (round-to-nearest bf16 is within 2^-9
    of each element); the gradients are bit-identical on a second call and
    the pad columns of dW keep their contents."""
    note(f"gate/up wgrad entry m={m} d={d} h={h} pads={pab},{px},{pw}")
    g = gen(11)
    dab = randn((m, h + pab), g, torch.bfloat16, cuda)
    dbb = randn((m, h + pab), g, torch.bfloat16, cuda)
    xb = randn((m, d + px), g, torch.bfloat16, cuda)
    da, db, x = dab[:, :h], dbb[:, :h], xb[:, :d]
    dwg, dwu = _wgrad(da, db, x, d + pw)
    ref_g, ref_u = np64(da).T @ np64(x), np64(db).T @ np64(x)
    assert on.rel_err(np64(dwg[:, :d]), ref_g) < 2.0 ** -8
    assert on.rel_err(np64(dwu[:, :d]), ref_u) < 2.0 ** -8
    if pw:
        assert bool((dwg[:, d:] == 7.0).all()) and bool((dwu[:, d:] == 7.0).all())
    dwg2, dwu2 = _wgrad(da, db, x, d + pw)
    assert torch.equal(dwg, dwg2) and torch.equal(dwu, dwu2)


def test_gate_up_wgrad_entry_without_tokens_zeroes(cuda):
    note("gate/up wgrad entry m=0")
    e = torch.empty((0, 64), dtype=torch.bfloat16, device=cuda)
    x = torch.empty((0, 32), dtype=torch.bfloat16, device=cuda)
    dwg, dwu = _wgrad(e, e, x, 40)
    assert bool((dwg[:, :32] == 0).all()) and bool((dwu[:, :32] == 0).all())
    assert bool((dwg[:, 32:] == 7.0).all())


def _bwd(da, db, x, wg, wu, dt, want=(True, True, True)):
    """nf_gemm_swiglu_bwd on row-strided views, its gradients (or None) in `dt`
    in buffers of NaN, and its workspace's size."""
    m, h = da.shape
    d = wg.shape[1]
    out = [torch.full(s, float("nan"), dtype=dt, device=wg.device) if k else None
           for s, k in zip(((m, d), (h, d), (h, d)), want)]
    L, code, dc = _lib.lib(), _lib.dtype_code(torch.bfloat16), _lib.dtype_code(dt)
    nb = L.nf_gemm_swiglu_bwd_workspace(m, d, h, *want)
    ws = torch.full((max(nb, 1),), 255, dtype=torch.uint8, device=wg.device)
    _lib.check(L.nf_gemm_swiglu_bwd(da.data_ptr(), db.data_ptr(), da.stride(0), x.data_ptr(),
                                    x.stride(0), wg.data_ptr(), wg.stride(0), wu.data_ptr(),
                                    wu.stride(0), _lib.ptr(out[0]), dc, _lib.ptr(out[1]),
                                    _lib.ptr(out[2]), dc, m, d, h, code, ws.data_ptr(), nb,
                                    _lib.stream_of(wg)), "nf_gemm_swiglu_bwd")
    torch.cuda.synchronize()
    return out, nb


def _bwd_inputs(m, d, h, pad, dev, seed):
    """da, db, x, w_gate, w_up as views whose rows end in `pad` NaN (w_up: twice)."""
    g = gen(seed)

    def view(rows, cols, extra, std=1.0):
        t = torch.full((rows, cols + extra), float("nan"), dtype=torch.bfloat16)
        t[:, :cols] = randn((rows, cols), g, torch.bfloat16, "cpu", std=std)
        return t.to(dev)[:, :cols]

    return [view(m, h, pad), view(m, h, pad), view(m, d, pad), view(h, d, pad, d ** -0.5),
            view(h, d, 2 * pad, d ** -0.5)]


# tile edges (256) and remainders, slices of dx's K across the seam between the
# gate and the up units (an odd number of 64-deep stages each), more than 8 dx
# slices, ragged last slices of both products, rows that are not whole vectors
# (padded copies: a workspace for both products whether split or not), strides
# that are not (element-wise copies and stores), one token, one unit
@pytest.mark.parametrize("m,d,h,pad,sx,sw", [
    (256, 256, 256, 0, True, False), (257, 264, 328, 8, True, False),
    (40, 72, 4104, 0, True, False), (3000, 136, 264, 8, True, True),
    (700, 200, 1000, 16, True, True), (300, 37, 101, 3, True, True),
    (1100, 36, 700, 0, True, True), (1, 8, 8, 0, False, False), (513, 520, 1, 7, True, True),
    (257, 263, 1001, 2, True, True), (3000, 255, 257, 0, True, True), (1, 1, 1, 0, True, True),
    (300, 72, 136, 3, False, False)])
def test_gate_up_bwd_entry_matches_fp64(cuda, m, d, h, pad, sx, sw):
    """dx = da W_gate + db W_up, dW_gate = da^T x, dW_up = db^T x in fp32 from the
    same bf16 operands in fp64, element by element; a second call gives the
    same bits, and bf16 results are the fp32 ones rounded once."""
    note(f"gate/up bwd entry m={m} d={d} h={h} pad={pad}")
    ops = _bwd_inputs(m, d, h, pad, cuda, m + d)
    da, db, x, wg, wu = (t.double() for t in ops)
    L = _lib.lib()
    assert (L.nf_gemm_swiglu_bwd_workspace(m, d, h, 1, 0, 0) > 0) == sx
    assert (L.nf_gemm_swiglu_bwd_workspace(m, d, h, 0, 1, 0) > 0) == sw
    got, _ = _bwd(*ops, torch.float32)
    want = [da @ wg + db @ wu, da.T @ x, db.T @ x]
    size = [da.abs() @ wg.abs() + db.abs() @ wu.abs(), da.abs().T @ x.abs(), db.abs().T @ x.abs()]
    # an accumulator takes K / 16 MFMAs of a few roundings each (4 are taken),
    # each 2^-24 of at most the sum of the products' sizes, then the slices' sum
    for v, w, z, k in zip(got, want, size, (2 * (h + 64), m + 64, m + 64)):
        assert ((v.double() - w).abs() <= (k / 4 + 33) * 2.0 ** -24 * z).all()
    again, _ = _bwd(*ops, torch.float32)
    half, _ = _bwd(*ops, torch.bfloat16)
    for v, a, b in zip(got, again, half):
        assert torch.equal(v, a) and torch.equal(v.bfloat16(), b)


@pytest.mark.parametrize("d,h", [(200, 1000), (201, 1003)])
@pytest.mark.parametrize("want", [(True, False, False), (False, True, False), (False, False, True),
                                  (True, True, False), (False, True, True), (False, False, False)])
def test_gate_up_bwd_entry_writes_what_is_wanted(cuda, want, d, h):
    """Any subset of the gradients: the values of a call for all three (their K
    split may differ: an fp32 sum in another order)."""
    m = 700
    note(f"gate/up bwd entry subset {want} d={d} h={h}")
    ops = _bwd_inputs(m, d, h, 0, cuda, 5)
    every, _ = _bwd(*ops, torch.float32)
    got, _ = _bwd(*ops, torch.float32, want)
    for v, e, k in zip(got, every, want):
        assert (v is not None) == k
        if k:
            assert (v - e).norm() <= 1e-6 * e.norm()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
def test_gate_up_bwd_entry_without_tokens_zeroes(cuda, dt):
    note(f"gate/up bwd entry m=0 {dt}")
    ops = _bwd_inputs(0, 40, 24, 0, cuda, 6)
    (dx, dwg, dwu), _ = _bwd(*ops, dt)
    assert dx.numel() == 0 and (dwg == 0).all() and (dwu == 0).all()


def test_gate_up_fwd_bwd_replays_in_a_graph(cuda):
    """The encoder-MLP gate/up step (GEMM with the SwiGLU epilogue, SwiGLU
    backward, split-K weight gradients with their transposes and reduce, dx)
    captured in a HIP graph: every replay matches the eager step bit for bit."""
    from tests.helpers import assert_graph_replays_match

    note("gate/up graph replay m=9408 d=384 h=1536")
    x, wg, wu, dact = _inputs(9408, 384, 1536, torch.bfloat16, cuda, seed=12)

    def make():
        leaves = [t.detach().requires_grad_(True) for t in (x, wg, wu)]

        def step():
            act = fused_gate_up_swiglu(*leaves)
            return (act, *torch.autograd.grad(act, leaves, dact))

        return step

    assert_graph_replays_match(make)


def test_gate_up_large_fwd_bwd_replays_in_a_graph(cuda):
    """The same for products above the line of nf_gemm_swiglu_bwd_wins, whose dx
    is two library GEMMs."""
    from tests.helpers import assert_graph_replays_match

    m, d, h = 2048, 4096, 8192
    note(f"gate/up graph replay m={m} d={d} h={h}")
    assert not _lib.lib().nf_gemm_swiglu_bwd_wins(m, d, h, 1)
    x, wg, wu, dact = _inputs(m, d, h, torch.bfloat16, cuda, seed=13)

    def make():
        leaves = [t.detach().requires_grad_(True) for t in (x, wg, wu)]

        def step():
            act = fused_gate_up_swiglu(*leaves)
            return (act, *torch.autograd.grad(act, leaves, dact))

        return step

    assert_graph_replays_match(make)
