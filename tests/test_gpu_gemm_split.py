"""The fp32 GEMM on three bf16 parts per operand (GPU, through nf_gemm_nt),
element by element against float64.

Bound: an accumulator takes K / 32 MFMA steps, each rounding it a few times
(4 is taken) to 2^-24 of at most sum |a b|; the products left out and the
final add are below 8 * 2^-24 of it.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from nuvla_forge_amd import _lib, _measure
from tests.helpers import gen, note, np64

pytestmark = pytest.mark.gpu


def _gemm(a, b, k):
    c = torch.full((a.shape[0], b.shape[0]), float("nan"), device=a.device)
    L = _measure.lib()
    _lib.check(L.nf_gemm_nt(a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0), c.data_ptr(),
                            c.stride(0), c.shape[0], c.shape[1], k, 0, _lib.stream_of(a)),
               "nf_gemm_nt")
    torch.cuda.synchronize()
    return c


# tile edges (256 x 128, 32-deep stages), remainders, rows that are not whole
# vectors (register copies element by element), one element
@pytest.mark.parametrize("m,n,k", [(256, 128, 32), (257, 129, 36), (255, 127, 64), (40, 300, 1000),
                                   (513, 260, 37), (3, 5, 1), (1, 1, 4), (300, 128, 4100)])
@pytest.mark.parametrize("scaled", [False, True])
def test_split_gemm_is_within_its_bound(cuda, m, n, k, scaled):
    note(f"split gemm m={m} n={n} k={k} scaled={scaled}")
    g = gen(m + 3 * n + 7 * k)
    a, b = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g)
    if scaled:  # magnitudes over 2^-30 .. 2^30 within each row
        a = a * 2.0 ** torch.randint(-30, 31, (m, k), generator=g)
        b = b * 2.0 ** torch.randint(-30, 31, (n, k), generator=g)
    a, b = a.to(cuda), b.to(cuda)
    got, A, B = np64(_gemm(a, b, k)), np64(a), np64(b)
    bound = (4 * (k / 32 + 1) + 8) * 2.0 ** -24 * (np.abs(A) @ np.abs(B).T)
    assert (np.abs(got - A @ B.T) <= bound).all()


def test_split_gemm_of_exact_products_is_exact(cuda):
    """24-bit operands whose products are exact: one term per output."""
    note("split gemm: exact values")
    vals = torch.tensor([1.0, 1 + 2.0 ** -23, 2 - 2.0 ** -23, -(2.0 ** 100) * (1 + 2.0 ** -12),
                         torch.finfo(torch.float32).max, torch.finfo(torch.float32).min, 0.0],
                        device=cuda)
    a = torch.zeros(len(vals), 64, device=cuda)
    a[:, 33] = vals
    b = torch.zeros(3, 64, device=cuda)
    b[:, 33] = torch.tensor([1.0, -0.5, 0.0], device=cuda)
    want = vals[:, None] * torch.tensor([1.0, -0.5, 0.0], device=cuda)
    assert torch.equal(_gemm(a, b, 64), want)


def test_split_gemm_keeps_infinities_and_nan(cuda):
    note("split gemm: inf and nan")
    inf, nan = float("inf"), float("nan")
    a = torch.ones(4, 32, device=cuda)
    a[0, 5], a[1, 5], a[2, 5] = inf, -inf, nan
    b = torch.full((2, 32), 0.5, device=cuda)
    got = _gemm(a, b, 32).cpu()
    assert (got[0] == inf).all() and (got[1] == -inf).all() and got[2].isnan().all()
    assert (got[3] == 16.0).all()


def test_split_gemm_of_infinities_and_the_smallest_values(cuda):
    """An infinity times any value but zero is an infinity, also where the value
    is below the last subnormal of the parts' type (2^-133)."""
    note("split gemm: inf times subnormals")
    inf = float("inf")
    a = torch.zeros(2, 32, device=cuda)
    a[0, 9], a[1, 9] = inf, -inf
    vals = torch.tensor([2.0 ** -126, 3 * 2.0 ** -134, 2.0 ** -134, 2.0 ** -140, -(2.0 ** -149),
                         2.0 ** -149, 0.0, -1.0], device=cuda)
    b = torch.zeros(len(vals), 32, device=cuda)
    b[:, 9] = vals
    got = _gemm(a, b, 32)
    want = torch.tensor([inf, -inf], device=cuda)[:, None] * vals
    assert torch.equal(got.isnan(), want.isnan()) and want.isnan().sum() == 2
    assert torch.equal(got.nan_to_num(), want.nan_to_num())


# Each operand in turn with parts that leave the most out: beside an exact
# leading part, a second and a third part of the largest size and one sign
@pytest.mark.parametrize("v", [1 + 2.0 ** -7 - 2.0 ** -15 + 2.0 ** -16 - 2.0 ** -23,
                               1 + 2.0 ** -8 + 2.0 ** -16 + 2.0 ** -17, 2 - 2.0 ** -23,
                               1 + 2.0 ** -7 - 2.0 ** -16 - 2.0 ** -23])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -90, 2.0 ** -112])
def test_split_gemm_of_operands_that_leave_the_most_out(cuda, v, scale):
    """Eight equal products: 2^-22 of them left out, 4 roundings of 2^-24, and
    2^-134 of each operand lost below 2^-110."""
    note(f"split gemm: large remainders {v!r} x {scale}")
    a, b = torch.zeros(5, 32, device=cuda), torch.zeros(7, 32, device=cuda)
    a[:, 4:12], b[:, 4:12] = v * scale, v
    got, A, B = np64(_gemm(a, b, 32)), np64(a), np64(b)
    bound = 8 * 2.0 ** -24 * (A @ B.T) + 8 * 2.0 ** -134 * v
    assert (np.abs(got - A @ B.T) <= bound).all()


# signalling NaNs, positive and negative, whose payload lies in the 16 bits
# below the first part
@pytest.mark.parametrize("bits", [0x7f800001, 0x7f80ffff, 0xff800001 - (1 << 32)])
def test_split_gemm_keeps_nan_payloads_nan(cuda, bits):
    note(f"split gemm: nan bits {bits:#x}")
    a = torch.ones(3, 32, device=cuda)
    a.view(torch.int32)[1, 7] = bits
    b = torch.full((2, 32), 0.5, device=cuda)
    got = _gemm(a, b, 32).cpu()
    assert got[1].isnan().all()
    assert (got[0] == 16.0).all() and (got[2] == 16.0).all()
