"""The elementwise ends of the distance scores' gradients: pkm_idw_grad_finish
and pkm_row_sumsq, in both layouts, at widths of one vector, a ragged share of
a lane group and several steps. The finish rounds step by step as the torch
expression does: the same bits. The sums of squares against float64 with the
bound of a float32 sum in any order, dim * 2^-24 of the sum.
"""
from __future__ import annotations

import pytest
import torch

from modelos_amd import product_keys as pk
from tests.helpers import gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,dim", [(1, 1, 4), (2, 17, 64), (8, 33, 128), (6, 5, 260), (3, 1000, 20)])
@pytest.mark.parametrize("row_major", [False, True])
def test_finish_and_sumsq(device, B, T, dim, row_major):
    g = gen(B + T)
    P = torch.randn((B, T, dim), generator=g).to(device)
    x = torch.randn((T, B, dim) if row_major else (B, T, dim), generator=g).to(device)
    s = torch.randn((B, T), generator=g).to(device)
    xb = x.transpose(0, 1) if row_major else x
    out = pk._idw_finish(P, x, s, row_major)
    expect = 2.0 * (P - xb * s[:, :, None])
    assert torch.equal(out.transpose(0, 1) if row_major else out, expect)
    q = pk._row_sumsq(x, row_major)
    e = xb.double().square().sum(-1)
    assert q.shape == (B, T) and ((q.double() - e).abs() <= e * dim * 2.0**-24).all()
    # rows that are not whole vectors take the torch expression: the same values
    if dim > 4:
        y, R = x[..., :-1], P[..., :-1]
        o = pk._idw_finish(R, y, s, row_major)
        yb = y.transpose(0, 1) if row_major else y
        assert torch.equal(o.transpose(0, 1) if row_major else o, 2.0 * (R - yb * s[:, :, None]))


def test_long_and_empty_rows(device):
    """Rows of 4 MB are the kernels' too; rows of no length are zeros."""
    B, T, dim = 2, 3, 1 << 20
    P = torch.randn((B, T, dim), device=device)
    x = torch.randn((T, B, dim), device=device)
    s = torch.randn((B, T), device=device)
    out = pk._idw_finish(P, x, s, True)
    assert torch.equal(out.transpose(0, 1), 2.0 * (P - x.transpose(0, 1) * s[:, :, None]))
    q = pk._row_sumsq(x, True)
    e = x.transpose(0, 1).double().square().sum(-1)
    assert ((q.double() - e).abs() <= e * dim / 16 * 2.0**-24).all()  # 16 chains a row
    assert torch.equal(pk._row_sumsq(x[..., :0].contiguous(), True), torch.zeros((B, T), device=device))


@pytest.mark.parametrize("B,T,row_major", [(2, (1 << 23) + 5, True), (1, (1 << 28) + 3, False)])
def test_sumsq_of_more_rows_than_a_grid(device, B, T, row_major):
    """Rows past one round of the grid, and past the 2^32 threads that 16 lanes
    for each row would be. Whole numbers: exact sums."""
    shape = (T, B, 4) if row_major else (B, T, 4)
    x = torch.randint(-8, 9, shape, device=device, dtype=torch.int8).float()
    q = pk._row_sumsq(x, row_major)
    expect = (x * x).sum(-1)
    assert torch.equal(q, expect.t() if row_major else expect)
    del x, q, expect
    torch.cuda.empty_cache()
