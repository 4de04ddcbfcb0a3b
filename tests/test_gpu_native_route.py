"""The ops' C++ host side against their general path (GPU).

The public functions give the plain call to ``_native`` and any other to the
autograd Functions in Python.  Both launch the same kernels, so every form is
held to the same bits; what makes a call not plain is answered ``None`` and
behaves as the Functions always did.
"""

from __future__ import annotations

from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest
import torch

from nuvla_forge_amd import _lib
from nuvla_forge_amd.kernels import (adaln_rmsnorm, chunked_ce, chunked_cross_entropy,
                                     fused_adaln_residual_rmsnorm, fused_gate_up_swiglu,
                                     fused_swiglu, swiglu)
from tests.helpers import gen, note, randn

pytestmark = pytest.mark.gpu

BF16, F32, F16 = torch.bfloat16, torch.float32, torch.float16


def _seam_inputs(dev, xd, yd, b=3, t=5, n=264, pad=8):
    """Conditioning as chunk views, a broadcast scale, row-strided x."""
    g = gen(3)
    x = randn((b * t, n + pad), g, xd, dev)[:, :n]
    y = randn((b * t, n), g, yd, dev)
    cond = randn((b, 6 * n), g, yd, dev, std=0.1).chunk(6, dim=-1)
    scale = randn((1, n), g, yd, dev, std=0.1).expand(b, n)
    w = randn((n,), g, xd, dev, std=0.02, mean=1.0)
    up = [randn((b * t, n), g, xd, dev), randn((b * t, n), g, xd, dev)]
    return [x, y, cond[2], w, scale, cond[0]], up, t


def _grads(fn, inputs, need, up):
    leaves = [v.detach().requires_grad_(k) for v, k in zip(inputs, need)]
    outs = fn(*leaves)
    outs = outs if isinstance(outs, tuple) else (outs,)
    want = [v for v in leaves if v.requires_grad]
    used = [(o, u) for o, u in zip(outs, up) if u is not None]
    got = torch.autograd.grad([o for o, _ in used], want, [u for _, u in used])
    return [*(o.detach() for o in outs), *got]


def _same(a, b):
    assert len(a) == len(b)
    for p, q in zip(a, b):
        assert p.dtype == q.dtype and p.shape == q.shape and torch.equal(p, q)


@pytest.mark.parametrize("xd,yd", [(BF16, BF16), (F32, BF16), (F32, F32), (F16, F16)])
@pytest.mark.parametrize("need", [(True,) * 6, (True, False, False, True, False, True)])
@pytest.mark.parametrize("drop", [None, 0, 1])
def test_seam_route_matches_the_function(cuda, xd, yd, need, drop):
    note(f"native seam {xd}/{yd} need={need} drop={drop}")
    inputs, up, t = _seam_inputs(cuda, xd, yd)
    if drop is not None:
        up[drop] = None
    assert _lib.native().seam(*inputs, t, 1e-6) is not None
    fast = _grads(lambda *v: fused_adaln_residual_rmsnorm(*v, tokens_per_sample=t), inputs, need, up)
    slow = _grads(lambda *v: adaln_rmsnorm._FusedAdaLNResidualRMSNorm.apply(*v, t, 1e-6), inputs,
                  need, up)
    _same(fast, slow)


@pytest.mark.parametrize("dtype", [BF16, F32, F16])
def test_swiglu_route_matches_the_function(cuda, dtype):
    note(f"native swiglu {dtype}")
    g = gen(4)
    a = randn((37, 3, 50), g, dtype, cuda).transpose(0, 1)  # not contiguous
    b = randn((3, 37, 50), g, dtype, cuda)
    up = [randn((3, 37, 50), g, dtype, cuda)]
    assert _lib.native().swiglu(a, b) is not None
    for need in ((True, True), (False, True)):
        _same(_grads(fused_swiglu, [a, b], need, up),
              _grads(swiglu._FusedSwiGLU.apply, [a, b], need, up))


@pytest.mark.parametrize("hd,wd,autocast", [(BF16, BF16, False), (F32, F32, True),
                                            (BF16, F32, True), (F32, F32, False),
                                            (F16, F32, False)])
def test_ce_route_matches_the_function(cuda, hd, wd, autocast):
    note(f"native ce {hd}/{wd} autocast={autocast}")
    g = gen(5)
    hid, w = randn((70, 40), g, hd, cuda), randn((333, 40), g, wd, cuda, std=0.1)
    tgt = torch.randint(0, 333, (70,), generator=g)
    tgt[::6] = -1
    tgt = tgt.to(cuda)
    up = [torch.tensor(0.7, device=cuda)]
    with torch.autocast("cuda", dtype=BF16, enabled=autocast):
        code = _lib.dtype_code(chunked_ce._compute_dtype(hid, w))
        assert _lib.native().ce(hid, w, tgt, 32, -1, code) is not None
        fast = _grads(lambda h, v: chunked_cross_entropy(h, v, tgt, 32, -1), [hid, w],
                      (True, True), up)
        slow = _grads(lambda h, v: chunked_ce._ChunkedCrossEntropy.apply(h, v, tgt, 32, -1, False),
                      [hid, w], (True, True), up)
    _same(fast, slow)


@pytest.mark.parametrize("index", [np.int64(7), torch.tensor(7), 7.0])
def test_ce_ignore_index_that_is_no_python_int(cuda, index):
    """A class of the vocabulary masked by an index of another type: what the
    plain int gives, to the bit, and the native entry answers None."""
    note(f"native ce ignore_index {index!r}")
    g = gen(9)
    hid, w = randn((64, 40), g, F32, cuda), randn((50, 40), g, F32, cuda)
    tgt = torch.randint(0, 50, (64,), generator=g)
    tgt[::3] = 7
    tgt = tgt.to(cuda)
    assert _lib.native().ce(hid, w, tgt, 16, index, 0) is None
    assert _lib.native().ce(hid, w, tgt, np.int64(16), 7, 0) is None
    up = [torch.tensor(1.0, device=cuda)]
    want = _grads(lambda h, v: chunked_cross_entropy(h, v, tgt, 16, 7), [hid, w], (True, True), up)
    for chunk in (16, np.int64(16)):
        got = _grads(lambda h, v: chunked_cross_entropy(h, v, tgt, chunk, index), [hid, w],
                     (True, True), up)
        _same(got, want)
    assert (want[1][::3] == 0).all()  # the masked rows have no gradient


@pytest.mark.parametrize("xd,gd,ud", [(BF16, BF16, BF16), (F32, F32, F32), (F32, BF16, F32)])
@pytest.mark.parametrize("need", [(True, True, True), (True, False, False), (False, False, True)])
def test_gate_up_route_matches_the_function(cuda, xd, gd, ud, need):
    note(f"native gate/up {xd}/{gd}/{ud} need={need}")
    g = gen(6)
    x, wg, wu = (randn((300, 136), g, xd, cuda), randn((264, 136), g, gd, cuda, std=0.1),
                 randn((264, 136), g, ud, cuda, std=0.1))
    up = [randn((300, 264), g, BF16, cuda)]
    assert _lib.native().gate_up(x, wg, wu) is not None
    with torch.autocast("cuda", dtype=BF16):
        _same(_grads(fused_gate_up_swiglu, [x, wg, wu], need, up),
              _grads(swiglu._FusedGateUpSwiGLU.apply, [x, wg, wu], need, up))


@pytest.mark.parametrize("xd,gd,ud", [
    (torch.float64,) * 3, (torch.int64, F32, F32), (F32, torch.float64, F32), (F32, F16, F32),
    (F32, F16, BF16), (BF16, F32, F16), (F16, F16, F16), (F32, BF16, F32)])
@pytest.mark.parametrize("need", [(True, True, True), (False, True, False), (False, False, True)])
def test_gate_up_gradients_in_any_input_types(cuda, xd, gd, ud, need):
    """Each gradient is the fp32 one rounded once to its own input's type: of
    no other input's type (an fp16 weight beside a bf16 or fp32 one must not
    overflow the other's gradient), and in types no kernel writes."""
    note(f"gate/up gradient types {xd}/{gd}/{ud} need={need}")
    g = gen(10)
    x = torch.randint(-8, 9, (70, 72), generator=g).to(cuda)  # whole in every type
    w = [torch.randint(-16, 17, (48, 72), generator=g).to(cuda) / 64 for _ in range(2)]
    need = (need[0] and xd.is_floating_point, *need[1:])
    # beyond fp16's range in the weight gradients
    up = [randn((70, 48), g, BF16, cuda, std=1e4)]
    with torch.autocast("cuda", dtype=BF16):
        want = _grads(fused_gate_up_swiglu, [x.float(), *w], need, up)
        got = _grads(fused_gate_up_swiglu, [x.to(xd), w[0].to(gd), w[1].to(ud)], need, up)
    types = [BF16, *(t for t, k in zip((xd, gd, ud), need) if k)]
    assert max(v.abs().max() for v in want[1:]) > torch.finfo(F16).max
    _same(got, [v.to(t) for v, t in zip(want, types)])


@pytest.mark.parametrize("which", ["x offset", "x stride", "w_gate offset", "w_up stride", "all"])
def test_gate_up_backward_of_views_off_vector_alignment(cuda, which):
    """Row-strided bf16 views whose rows do not start on 16 bytes: the same bits as
    contiguous copies of them, from both hosts."""
    note(f"gate/up views {which}")
    m, d, h = 300, 72, 136
    g = gen(14)

    def view(name, rows):
        wide = randn((rows, d + 16), g, BF16, cuda, std=1.0 if name == "x" else d ** -0.5)
        off = 1 if which in (f"{name} offset", "all") else 0
        if which == f"{name} stride":
            wide = wide[:, :d + 3].contiguous()
        return wide[:, off:off + d]

    inputs = [view("x", m), view("w_gate", h), view("w_up", h)]
    assert any(v.data_ptr() % 16 or v.stride(0) % 8 for v in inputs)
    up = [randn((m, h), g, BF16, cuda)]

    def run(fn, ops):
        leaves = [v.detach().requires_grad_(True) for v in ops]  # keeps strides
        out = fn(*leaves)
        return [out.detach(), *torch.autograd.grad(out, leaves, up)]

    got = run(fused_gate_up_swiglu, inputs)
    _same(got, run(swiglu._FusedGateUpSwiGLU.apply, inputs))
    want = run(fused_gate_up_swiglu, [v.contiguous().clone() for v in inputs])
    for a, e in zip(got[1:], want[1:]):
        assert (a.double() - e.double()).norm() <= 2.0 ** -7 * e.double().norm()


@pytest.mark.parametrize("m,d,h,need", [
    (2056, 4096, 8200, (True, True, True)), (2056, 4096, 8200, (True, False, False)),
    (2056, 4096, 8200, (False, True, True)), (2056, 4096, 8200, (True, False, True)),
    (8197, 72, 136, (True, False, False)), (8200, 37, 101, (True, False, False))])
def test_gate_up_large_products(cuda, m, d, h, need):
    """Beyond the line of nf_gemm_swiglu_bwd_wins (dx alone: from 8192 tokens): both
    hosts alike, and each gradient against fp32 products of the same bf16 inputs."""
    note(f"gate/up large m={m} d={d} h={h} need={need}")
    assert not _lib.lib().nf_gemm_swiglu_bwd_wins(m, d, h, any(need[1:]))
    g = torch.Generator(device=cuda).manual_seed(12)
    rnd = lambda *s, std=1.0: torch.randn(*s, device=cuda, generator=g).mul_(std).bfloat16()  # noqa: E731
    inputs = [rnd(m, d), rnd(h, d, std=d ** -0.5), rnd(h, d, std=d ** -0.5)]
    up = [rnd(m, h)]
    got = _grads(fused_gate_up_swiglu, inputs, need, up)
    _same(got, _grads(swiglu._FusedGateUpSwiGLU.apply, inputs, need, up))
    f = lambda x, wg, wu: torch.nn.functional.silu(x @ wg.T) * (x @ wu.T)  # noqa: E731
    want = _grads(f, [v.float() for v in inputs], need, [up[0].float()])
    # a, b, da, db, act, dx's partial sum and the gradients are rounded to bf16
    # (2^-9 of each at most, about half that in the norm), at most five of
    # them in a row and independent: sqrt(5) 2^-9
    for a, e in zip(got, want):
        assert a.dtype == BF16
        assert (a.float() - e).norm() <= 5 ** 0.5 * 2.0 ** -9 * e.norm()


@pytest.mark.parametrize("m,d,h", [(300, 136, 264), (5, 64, 1000), (300, 36, 100)])
@pytest.mark.parametrize("dtype", [BF16, F32])
def test_gate_up_without_a_backward(cuda, m, d, h, dtype):
    """No backward to come (no_grad, or no input that wants a gradient): only
    act is written; the forward of a training step is the reference, one bf16
    rounding (an ulp, 2^-7, at most) apart."""
    note(f"native gate/up inference m={m} d={d} h={h} {dtype}")
    g = gen(8)
    x = randn((m, d), g, dtype, cuda)
    w = [randn((h, d), g, dtype, cuda, std=d ** -0.5).requires_grad_(True) for _ in range(2)]
    with torch.autocast("cuda", dtype=BF16):
        want = fused_gate_up_swiglu(x, *w)
        assert want.requires_grad
        with torch.no_grad():
            got = [fused_gate_up_swiglu(x, *w)]
        with torch.inference_mode():
            got.append(fused_gate_up_swiglu(x, *w))
        got.append(fused_gate_up_swiglu(x, *(v.detach() for v in w)))
    ref = want.detach().float()
    for act in got:
        assert act.dtype == BF16 and act.shape == (m, h) and not act.requires_grad
        assert ((act.float() - ref).abs() <= 2.0 ** -7 * ref.abs() + 1e-5).all()


def test_saved_tensors_go_through_the_hooks(cuda):
    note("native route under saved-tensor hooks")
    inputs, up, t = _seam_inputs(cuda, F32, BF16)
    plain = _grads(lambda *v: fused_adaln_residual_rmsnorm(*v, tokens_per_sample=t), inputs,
                   (True,) * 6, up)
    packed = []

    def pack(v):
        packed.append(v.shape)
        return v.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda v: v.to(cuda)):
        hooked = _grads(lambda *v: fused_adaln_residual_rmsnorm(*v, tokens_per_sample=t), inputs,
                        (True,) * 6, up)
    assert len(packed) == 6
    _same(hooked[:2], plain[:2])
    for a, b in zip(hooked, plain):
        assert torch.equal(a, b)


def test_calls_that_are_not_plain_take_the_general_path(cuda):
    note("native route: what it leaves alone")
    g = gen(7)
    a, b = randn((4, 16), g, BF16, cuda), randn((4, 16), g, BF16, cuda)
    n = _lib.native()
    with torch.autograd.forward_ad.dual_level():  # forward mode stays refused
        dual = torch.autograd.forward_ad.make_dual(a, b)
        assert n.swiglu(dual, b) is None
        with pytest.raises(RuntimeError):
            fused_swiglu(dual, b)
    with pytest.raises(RuntimeError):  # and so does vmap
        torch.func.vmap(fused_swiglu)(a, b)

    class Tagged(torch.Tensor):
        pass

    assert n.swiglu(a.as_subclass(Tagged), b) is None
    assert n.swiglu(a, b.float()) is None and n.swiglu(a, b[:2]) is None
    assert n.swiglu(a.double(), b.double()) is None
    with pytest.raises(TypeError):
        fused_swiglu(a, b.float())
    x, y = randn((6, 8), g, BF16, cuda), randn((6, 8), g, BF16, cuda)
    c, w = randn((2, 8), g, BF16, cuda), randn((8,), g, BF16, cuda)
    assert n.seam(x, y, c, w, c, c, 3, 1e-6) is not None
    assert n.seam(x, y, c, w, c, c, 4, 1e-6) is None  # rows not whole samples
    with pytest.raises(ValueError):
        fused_adaln_residual_rmsnorm(x, y, c, w, c, c, 4)
    assert n.seam(x.t().contiguous().t(), y, c, w, c, c, 3, 1e-6) is None  # strided columns
    assert n.seam(x, y.float(), c, w, c, c, 3, 1e-6) is None  # 16-bit x with fp32 y
    assert n.seam(x, y.cpu(), c, w, c, c, 3, 1e-6) is None
    traced = torch.jit.trace(lambda p, q: fused_swiglu(p, q), (a, b), check_trace=False)
    assert torch.equal(traced(b, a), fused_swiglu(b, a))


def test_native_route_on_another_stream(cuda):
    note("native route on a side stream")
    inputs, up, t = _seam_inputs(cuda, BF16, BF16, b=4, t=64, n=1024, pad=0)
    want = _grads(lambda *v: fused_adaln_residual_rmsnorm(*v, tokens_per_sample=t), inputs,
                  (True,) * 6, up)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = _grads(lambda *v: fused_adaln_residual_rmsnorm(*v, tokens_per_sample=t), inputs,
                     (True,) * 6, up)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    _same(got, want)


def test_native_route_from_several_threads(cuda):
    """Four threads, a stream each, take turns at the interpreter while others
    are inside a call: each gets what a thread of its own gets."""
    note("native route from four threads")
    inputs, up, t = _seam_inputs(cuda, BF16, BF16, b=4, t=16, n=512, pad=0)

    def step():
        return _grads(lambda *v: fused_adaln_residual_rmsnorm(*v, tokens_per_sample=t), inputs,
                      (True,) * 6, up)

    want = step()
    torch.cuda.synchronize()

    def work(_):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            outs = [step() for _ in range(8)]
        stream.synchronize()
        return outs

    with ThreadPoolExecutor(4) as ex:
        for outs in ex.map(work, range(4)):
            for got in outs:
                _same(got, want)
