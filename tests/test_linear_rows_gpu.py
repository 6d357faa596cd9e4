"""pkm_linear_rows (a Linear over a few bf16 rows) against float64.

The value Linears of a decode step: row counts around the 16-row tiles, input
widths of fewer k-steps than waves, of a ragged share per wave and of many, one
tile of outputs and several, with and without a bias. Bound: one bf16 rounding
(2^-9 relative, 2^-8 with the bias of another magnitude) of float32 sums whose
error is far below it, taken relative to the sum of |terms|.
"""
from __future__ import annotations

import pytest
import torch

from modelos_amd import _lib
from modelos_amd.pkm import memory
from tests.helpers import gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("rows,fin,fout", [(1, 32, 16), (8, 1024, 1024), (15, 96, 48), (16, 288, 16), (17, 512, 1024),
                                           (33, 1056, 32), (64, 4096, 64)])
def test_against_float64(device, rows, fin, fout, bias):
    g = gen(rows + fin)
    lin = torch.nn.Linear(fin, fout, bias=bias)
    with torch.no_grad():
        lin.weight.copy_(torch.randn((fout, fin), generator=g) * fin**-0.5)
        if bias:
            lin.bias.copy_(torch.randn(fout, generator=g))
    lin = lin.to(device=device, dtype=torch.bfloat16)
    x = torch.randn((rows, fin), generator=g).to(torch.bfloat16).to(device)
    # (at the last size the layer calls the BLAS, which is the faster one there)
    takes = memory._rows_kernel_takes(x, lin.weight, lin.bias)
    assert takes == (rows <= 16 or fin <= 1056)
    y = torch.empty((rows, fout), dtype=torch.bfloat16, device=device)
    _lib.call("pkm_linear_rows", _lib.ptr(x), _lib.ptr(lin.weight), _lib.ptr(lin.bias), rows, fin, fout,
              _lib.dtype_code(x), _lib.ptr(y), _lib.stream_of(x.device))
    w64, x64 = lin.weight.detach().double(), x.double()
    b64 = lin.bias.detach().double() if bias else torch.zeros(fout, dtype=torch.float64, device=device)
    expect = x64 @ w64.t() + b64
    bound = (x64.abs() @ w64.abs().t() + b64.abs()) * 2.0**-20 + expect.abs() * 2.0**-8
    assert ((y.double() - expect).abs() <= bound).all()
    if takes:
        assert torch.equal(y, memory._linear(lin, x, True))


def test_what_it_does_not_take(device):
    lin = torch.nn.Linear(64, 32).to(device=device, dtype=torch.bfloat16)
    x = torch.randn((65, 64), device=device).to(torch.bfloat16)
    assert not memory._rows_kernel_takes(x, lin.weight, lin.bias)  # rows
    assert memory._rows_kernel_takes(x[:64], lin.weight, lin.bias)
    assert not memory._rows_kernel_takes(x[:8, ::2], lin.weight[:, :32], lin.bias)  # strides
    assert not memory._rows_kernel_takes(x[:8].float(), lin.weight.float(), lin.bias.float())
    assert not memory._rows_kernel_takes(x.reshape(-1)[1:8 * 64 + 1].view(8, 64), lin.weight, lin.bias)  # alignment
    assert not memory._rows_kernel_takes(x[:8], lin.weight, lin.bias[:1])  # a bias that broadcasts
    y = torch.empty((8, 32), dtype=torch.bfloat16, device=device)
    for rows, fin, fout, code in ((65, 64, 32, 1), (8, 48, 32, 1), (8, 64, 24, 1), (8, 64, 32, 0)):
        with pytest.raises(_lib.PkmError):
            _lib.call("pkm_linear_rows", _lib.ptr(x), _lib.ptr(lin.weight), None, rows, fin, fout, code, _lib.ptr(y),
                      _lib.stream_of(x.device))


# Sizes that the kernel does not take, or is the slower one at, go to F.linear.
def test_sizes_past_the_rule_run(device):
    for rows, fin, fout in ((3, 0, 16), (3, 32, 0), (17, 1088, 16), (16, 4128, 16), (2, 1 << 20, 16), (2, 64, 4112)):
        lin = torch.nn.Linear(fin, fout).to(device=device, dtype=torch.bfloat16) if fin and fout else None
        w = lin.weight if lin else torch.zeros((fout, fin), dtype=torch.bfloat16, device=device)
        b = lin.bias if lin else torch.ones(fout, dtype=torch.bfloat16, device=device)
        x = torch.randn((rows, fin), device=device).to(torch.bfloat16)
        assert not memory._rows_kernel_takes(x, w, b)
        y = memory._Linear.apply(x, w, b, True)
        assert torch.equal(y, torch.nn.functional.linear(x, w, b))


def test_infinities_and_nan(device):
    """An infinite or NaN row of x reaches its own row of y only, one of the
    weight its own column; rows past the last tile's are copies of the last."""
    rows, fin, fout = 9, 96, 32
    g = gen(77)
    x = torch.randn((rows, fin), generator=g).to(torch.bfloat16)
    w = torch.randn((fout, fin), generator=g).to(torch.bfloat16)
    x[2, 5], x[8, 95], w[17, 40] = float("inf"), float("nan"), float("-inf")
    lin = torch.nn.Linear(fin, fout)
    with torch.no_grad():
        lin.weight.copy_(w.float())
    lin = lin.to(device=device, dtype=torch.bfloat16)
    x = x.to(device)
    assert memory._rows_kernel_takes(x, lin.weight, lin.bias)
    y = memory._linear(lin, x, True).double()
    expect = x.double() @ lin.weight.detach().double().t() + lin.bias.detach().double()
    assert torch.equal(y.isnan(), expect.isnan())
    inf = expect.isinf()
    assert torch.equal(y[inf], expect[inf])
    fine = expect.isfinite()
    bound = expect.abs() * 2.0**-8 + fin * 2.0**-18
    assert ((y - expect).abs()[fine] <= bound[fine]).all()
