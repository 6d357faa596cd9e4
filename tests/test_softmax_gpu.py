"""GPU parity of the score softmax (pkm_softmax_fwd / pkm_softmax_bwd)
against the reference expression F.softmax(scores.float(), -1).type_as(scores)
(pkm/memory.py:218) and its autograd, run by torch on the same device. The
kernels sum in column order (torch's softmax in a reduction tree), so the
float32 results agree to rounding: 1e-5 (f32) / 2e-2 (bf16) relative."""
from __future__ import annotations

import pytest
import torch

from modelos_amd import _lib
from modelos_amd.product_keys import score_softmax
from tests.helpers import REL_TOL, assert_rel_close, gen

pytestmark = pytest.mark.gpu


def _run(fn, x, dy):
    xx = x.clone().requires_grad_(True)
    y = fn(xx)
    y.backward(dy)
    return y.detach(), xx.grad


def _ref(x):
    return torch.softmax(x.float(), dim=-1).type_as(x)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16], ids=["bf16", "f32", "f16"])
@pytest.mark.parametrize("shape", [(131072, 32), (300, 64), (77, 7), (5, 1), (3, 4, 33), (101, 8), (99, 16), (50, 4),
                                   (8192, 64 * 4), (33, 65), (7, 1000), (3, 5000), (31, 128), (13, 512)],
                         ids=["layer", "k64", "k7", "k1", "3d-k33", "k8", "k16", "k4", "fw-h4k64", "k65", "k1000",
                              "k5000", "k128", "k512"])
def test_matches_torch(device, dtype, shape):
    g = gen(11)
    x = (torch.randn(shape, generator=g) * 4).to(dtype).to(device)
    dy = torch.randn(shape, generator=g).to(dtype).to(device)
    y, dx = _run(score_softmax, x, dy)
    e_y, e_dx = _run(_ref, x, dy)
    torch.cuda.synchronize()
    assert y.dtype == dtype and dx.dtype == dtype
    assert_rel_close(y, e_y, REL_TOL[dtype], "y")
    assert_rel_close(dx, e_dx, REL_TOL[dtype], "dx")
    # rows sum to one (float32 probabilities before the rounding)
    sum_tol = {torch.bfloat16: 5e-2, torch.float16: 5e-3, torch.float32: 1e-5}[dtype]
    assert_rel_close(y.double().sum(-1), torch.ones(shape[:-1], dtype=torch.float64), sum_tol, "row sums")


def test_equal_and_extreme_scores(device):
    x = torch.tensor([[0.0] * 32, [1e4] + [-1e4] * 31, [float("-inf")] + [0.0] * 31], device=device)
    dy = torch.randn(x.shape, generator=gen(12)).to(device)
    y, dx = _run(score_softmax, x, dy)
    e_y, e_dx = _run(_ref, x, dy)
    torch.cuda.synchronize()
    assert_rel_close(y, e_y, 1e-6, "y")
    assert_rel_close(dx, e_dx, 1e-5, "dx")


def test_deterministic_and_limits(device):
    x = torch.randn((1000, 32), generator=gen(13)).to(torch.bfloat16).to(device)
    assert torch.equal(score_softmax(x), score_softmax(x))
    with pytest.raises(_lib.PkmError):
        y = torch.empty((2, 65537), device=device)
        _lib.call("pkm_softmax_fwd", _lib.ptr(y), 2, 65537, _lib.dtype_code(y), _lib.ptr(y), _lib.stream_of(y.device))
    with pytest.raises(NotImplementedError):
        score_softmax(torch.zeros((2, 4), dtype=torch.float64, device=device))


def test_long_rows_extreme_scores(device):
    """The wave-per-row kernel (rows longer than 64): equal scores, one
    dominant score, a -inf entry."""
    x = torch.zeros((3, 256), device=device)
    x[1, 0], x[1, 1:] = 1e4, -1e4
    x[2, 5] = float("-inf")
    dy = torch.randn(x.shape, generator=gen(14)).to(device)
    y, dx = _run(score_softmax, x, dy)
    e_y, e_dx = _run(_ref, x, dy)
    torch.cuda.synchronize()
    assert_rel_close(y, e_y, 1e-6, "y")
    assert_rel_close(dx, e_dx, 1e-5, "dx")


# dx = p (dy - <dy, p>) cancels where a row is close to one-hot: compared with
# float64 relative to the size of its terms, p (|dy| + <|dy|, p>). Bounds: one
# rounding of a 16-bit output (2^-8, 2^-11) and 64 float32 roundings (exp of a
# rounded difference, the sums over a row) of 2^-24 relative to the terms.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16], ids=["bf16", "f32", "f16"])
@pytest.mark.parametrize("shape", [(2, 24), (50, 24), (99, 16), (40, 128), (33, 65), (21, 256)], ids=str)
def test_gradient_relative_to_its_terms(device, dtype, shape):
    g = gen(15)
    x = (torch.randn(shape, generator=g) * 4).to(dtype).to(device)
    dy = torch.randn(shape, generator=g).to(dtype).to(device)
    y, dx = _run(score_softmax, x, dy)
    p = torch.softmax(x.double(), -1)
    d = dy.double()
    expect = p * (d - (d * p).sum(-1, keepdim=True))
    terms = p * (d.abs() + (d.abs() * p).sum(-1, keepdim=True))
    eps = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 0.0}[dtype] + 64 * 2.0**-24
    floor = 2.0**-24 if dtype == torch.float16 else 0.0  # its smallest subnormal
    assert ((dx.double() - expect).abs() <= eps * terms + floor).all()
    assert ((y.double() - p).abs() <= eps * p + floor).all()


def test_more_rows_than_a_grid_of_lane_groups(device):
    """2^28 + 3 rows of 64 float32 (64 GiB): 16 lanes a row would be more
    threads than a grid holds, so a lane takes a row. Equal scores: 1 / 64."""
    if torch.cuda.mem_get_info(device)[0] < 160 << 30:
        pytest.skip("needs 160 GiB of device memory")
    rows = (1 << 28) + 3
    x = torch.zeros((rows, 64), device=device)
    marked = torch.tensor([0, (1 << 28) - 1, 1 << 28, rows - 1], device=device)
    x[marked] = torch.arange(64, dtype=torch.float32, device=device) / 8
    y = torch.empty_like(x)
    _lib.call("pkm_softmax_fwd", _lib.ptr(x), rows, 64, _lib.dtype_code(x), _lib.ptr(y), _lib.stream_of(x.device))
    assert_rel_close(y[marked], torch.softmax(x[marked].double(), -1), 1e-6, "marked rows")
    y[marked] = 2.0**-6
    for a in range(0, rows, 1 << 26):
        assert bool((y[a:a + (1 << 26)] == 2.0**-6).all()), f"rows from {a}"
    del x, y
    torch.cuda.empty_cache()
