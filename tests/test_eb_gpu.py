"""Parity of the HIP embedding-bag kernels (through the C ABI) with the oracle.

Small and ragged sizes are compared element-wise with oracle/eb.py on the same
seeded inputs; the full standalone size (16384 bags x 128 lookups into a
2^20 x 1024 bf16 table) is checked on sampled bags / rows against the oracle
plus size-independent properties (column-sum checksum, untouched rows exactly
zero, bitwise run-to-run determinism). Tolerances: 1e-5 relative (fp32),
2e-2 (bf16), 2e-3 (fp16), relative to each tensor's scale.
"""
import pytest
import torch

from oracle import eb as ref
from tests.helpers import REL_TOL, assert_rel_close, eb_inputs

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]

# (B, L, K, D): row lengths hit every lane-group shape (LPG 1..64, VPL 1..8),
# bag sizes around the 64-entry batch, tiny and empty cases.
SHAPES = [
    (33, 17, 1000, 1024),
    (7, 64, 500, 512),
    (9, 65, 300, 256),
    (5, 128, 2000, 2048),
    (3, 3, 50, 4096),
    (17, 31, 100, 128),
    (21, 5, 64, 64),
    (4, 2, 10, 32),
    (6, 1, 9, 16),
    (2, 7, 40, 8),
]


def _dev(*ts, device):
    return [t.to(device) if t is not None else None for t in ts]


def _reduce_supported(D, dtype):
    """The backward / double-backward kernels hold a whole row per lane group:
    dim / (16 B / element size) must be LPG * VPL with VPL <= 8."""
    epv = 4 if dtype == torch.float32 else 8
    return (D // epv) <= 512


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("B,L,K,D", SHAPES)
def test_forward_parity(B, L, K, D, dtype, device):
    from modelos_amd import embedding_bag as eb

    if dtype == torch.float32 and D == 8:
        D = 12  # not a multiple of 8 for 16-bit, exercises fp32 LPG=1; 16-bit uses the scalar fallback below
    W, idx, p, _ = eb_inputs(B, L, K, D, dtype, seed=B * 1000 + L, with_grad=False)
    out = eb.eb_forward(*_dev(idx, W, p, device=device))
    assert out.dtype == dtype and out.shape == (B, D)
    assert_rel_close(out, ref.eb_forward(idx, W, p), REL_TOL[dtype], f"forward {dtype} {B,L,K,D}")


@pytest.mark.parametrize("D", [12, 20, 6])
def test_forward_scalar_fallback(D, device):
    from modelos_amd import embedding_bag as eb

    W, idx, p, _ = eb_inputs(5, 9, 30, D, torch.bfloat16, seed=D, with_grad=False)
    out = eb.eb_forward(*_dev(idx, W, p, device=device))
    assert_rel_close(out, ref.eb_forward(idx, W, p), 2e-2, "scalar fallback")


def test_forward_unweighted_mixed_dtypes_and_invalid(device):
    from modelos_amd import embedding_bag as eb

    W, idx, p, _ = eb_inputs(19, 40, 700, 1024, torch.bfloat16, seed=5, psw_dtype=torch.float32, with_grad=False)
    idx[0, 0] = -5
    idx[3, 39] = 700
    idx[7, 12] = 1 << 40
    dW, didx, dp = _dev(W, idx, p, device=device)
    assert_rel_close(eb.eb_forward(didx, dW, dp), ref.eb_forward(idx, W, p), 2e-2, "fp32 psw on bf16 table")
    assert_rel_close(eb.eb_forward(didx, dW, None), ref.eb_forward(idx, W, None), 2e-2, "unweighted")
    assert eb.count_invalid_indices(didx, 700) == 3


# The gather's layouts: whole rows with one to sixteen waves per bag (few bags;
# bag lengths around the 16-lookup steps), two bags a wave from 8192 bags on
# (an odd count), rows of 32 k and 16 k vectors. Row 0 holds infinities and is
# only looked up out of range: absent lookups, with NaN weights, add nothing.
@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("B,L,nvec", [(1, 256, 128), (8, 17, 64), (3, 1, 64), (40, 100, 128), (8193, 5, 64),
                                      (70, 33, 96), (70, 16, 48), (5, 300, 16)])
def test_forward_gather_layouts(B, L, nvec, dtype, device):
    from modelos_amd import embedding_bag as eb

    D = nvec * (4 if dtype == torch.float32 else 8)
    W, idx, p, _ = eb_inputs(B, L, 500, D, dtype, seed=B + L, with_grad=False)
    idx = idx.clamp_min(1)
    expect = ref.eb_forward(idx, W, p)
    if L > 2:
        p0 = p.clone()
        p0[:, 1] = 0
        expect = ref.eb_forward(idx, W, p0)
        idx[:, 1] = torch.where(torch.arange(B) % 2 == 0, -1, 500)
        p[:, 1] = float("nan")
    W[0] = float("inf")
    out = eb.eb_forward(*_dev(idx, W, p, device=device))
    cond = ref.eb_forward(idx.clamp(1, 499), W.abs(), p.abs().nan_to_num(0.0))
    assert_rel_close(out, expect, REL_TOL[dtype], f"forward {dtype} {B,L,D}", cond=cond)


# A step of the gather takes 16 lookups, a last one of at most 8 half of it:
# both sides of each line, with the lookups of a bag in one wave (2048 bags) and
# shared by several (2 bags). Row 0 holds infinities and is not looked up.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("L", [7, 8, 9, 15, 16, 17, 24, 25, 40, 41, 264, 265])
@pytest.mark.parametrize("B,nvec", [(2, 16), (2, 64), (2048, 32), (2048, 64)])
def test_forward_gather_last_step(B, nvec, L, dtype, device):
    from modelos_amd import embedding_bag as eb

    D = nvec * (4 if dtype == torch.float32 else 8)
    B = B if L < 100 else min(B, 300)
    W, idx, p, _ = eb_inputs(B, L, 300, D, dtype, seed=B + L, with_grad=False)
    idx = idx.clamp_min(1)
    W[0] = 0
    expect = ref.eb_forward(idx, W, p)
    cond = ref.eb_forward(idx, W.abs(), p.abs())
    W[0] = float("inf")
    out = eb.eb_forward(*_dev(idx, W, p, device=device))
    assert_rel_close(out, expect, REL_TOL[dtype], f"forward {dtype} {B,L,D}", cond=cond)


# More bags than one grid holds: two bags a wave, 16 slices of an 8 KB row, so
# 2^23 bags are 2^26 waves (two launches; 64 GiB of output). One lookup a bag and
# weights that are powers of two: the rows are exact.
def test_forward_more_bags_than_a_grid(device):
    from modelos_amd import embedding_bag as eb

    B, K, D = (1 << 23) + 3, 257, 4096
    if torch.cuda.mem_get_info(device)[0] < 100 << 30:
        pytest.skip("needs 100 GiB of device memory")
    gen = torch.Generator(device=device).manual_seed(5)
    W = torch.randn((K, D), generator=gen, device=device).to(torch.bfloat16)
    idx = torch.randint(0, K, (B, 1), generator=gen, device=device)
    p = torch.tensor([0.5, 1.0, 2.0], device=device)[torch.randint(0, 3, (B, 1), generator=gen, device=device)]
    out = eb.eb_forward(idx, W, p)
    for a in range(0, B, 1 << 20):
        rows = W[idx[a:a + (1 << 20), 0]]
        rows *= p[a:a + (1 << 20)].to(torch.bfloat16)
        assert torch.equal(out[a:a + (1 << 20)], rows), f"bags from {a}"
    del out, rows
    torch.cuda.empty_cache()


def test_forward_empty(device):
    from modelos_amd import embedding_bag as eb

    W = torch.randn(10, 64, device=device)
    assert eb.eb_forward(torch.zeros(0, 3, dtype=torch.long, device=device), W, None).shape == (0, 64)
    out = eb.eb_forward(torch.zeros(4, 0, dtype=torch.long, device=device), W, torch.zeros(4, 0, device=device))
    assert (out == 0).all()


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("B,L,K,D", SHAPES)
def test_backward_parity(B, L, K, D, dtype, device):
    from modelos_amd import embedding_bag as eb

    W, idx, p, g = eb_inputs(B, L, K, D, dtype, seed=B * 7 + L)
    if not _reduce_supported(D, dtype):
        from modelos_amd._lib import PkmError

        with pytest.raises(PkmError, match="not supported"):
            eb.eb_backward(*_dev(idx, W, p, g, device=device))
        return
    gW, gp = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    eW, ep = ref.eb_backward(idx, W, p, g)
    assert gW.dtype == dtype and gp.dtype == p.dtype
    assert_rel_close(gW, eW, REL_TOL[dtype], f"grad_weight {dtype} {B,L,K,D}")
    assert_rel_close(gp, ep, REL_TOL[dtype], f"grad_psw {dtype} {B,L,K,D}")


def _hot_indices(B, L, K, seed):
    """Indices with heavy rows: row 3 takes ~1/3 of all lookups, rows 4 and 5
    ~600 each (adjacent heavy rows share chunks), the rest uniform, plus a few
    out-of-range entries."""
    g = torch.Generator().manual_seed(seed)
    idx = torch.randint(0, K, (B, L), generator=g)
    u = torch.rand((B, L), generator=g)
    idx[u < 1 / 3] = 3
    flat = idx.view(-1)
    pos = torch.randperm(B * L, generator=g)
    flat[pos[:600]] = 4
    flat[pos[600:1200]] = 5
    flat[pos[1200:1205]] = -1
    return idx


# 97 bags: the sparse plan; 400: the general one, with two digits and with one.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("B,K", [(97, 5000), (400, 5000), (400, 200)])
@pytest.mark.parametrize("D", [1024, 64])
def test_backward_heavy_rows(D, B, K, dtype, device):
    from modelos_amd import embedding_bag as eb

    L = 64
    W, _, p, g = eb_inputs(B, L, K, D, dtype, seed=21)
    idx = _hot_indices(B, L, K, seed=22)
    gW, gp = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    eW, ep = ref.eb_backward(idx, W, p, g)
    # (row 3 of 400 bags sums 8500 terms of both signs: float32 roundings of sums in another order, up to
    # 2^-24 times the chunks' partial sums each, are bounded by the sum of |terms| and not by the result)
    cW = ref.eb_backward(idx, W.abs(), p.abs(), g.abs())[0] if B > 97 else None
    assert_rel_close(gW, eW, REL_TOL[dtype], "heavy grad_weight", cond=cW)
    assert_rel_close(gp, ep, REL_TOL[dtype], "heavy grad_psw")
    assert (gp.cpu()[idx < 0] == 0).all()


def test_backward_unweighted_and_deterministic(device):
    from modelos_amd import embedding_bag as eb

    W, idx, _, g = eb_inputs(64, 48, 3000, 512, torch.float32, seed=23, psw=False)
    idx = _hot_indices(64, 48, 3000, seed=24)
    dW, didx, dg = _dev(W, idx, g, device=device)
    gW1, gp1 = eb.eb_backward(didx, dW, None, dg)
    gW2, _ = eb.eb_backward(didx, dW, None, dg)
    assert gp1 is None
    eW, _ = ref.eb_backward(idx, W, None, g)
    assert_rel_close(gW1, eW, 1e-5, "unweighted grad_weight")
    assert torch.equal(gW1, gW2), "backward is not bitwise deterministic"


def test_backward_empty_bags_zero_grad(device):
    from modelos_amd import embedding_bag as eb

    W = torch.randn(100, 256, device=device)
    gW, gp = eb.eb_backward(
        torch.zeros(0, 4, dtype=torch.long, device=device), W, torch.zeros(0, 4, device=device),
        torch.zeros(0, 256, device=device),
    )
    assert (gW == 0).all() and gp.shape == (0, 4)


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("B,L,K,D", SHAPES)
@pytest.mark.parametrize("with_a", [True, False])
def test_double_backward_parity(B, L, K, D, dtype, with_a, device):
    from modelos_amd import embedding_bag as eb

    _, idx, a, g = eb_inputs(B, L, K, D, dtype, seed=B + L + D, psw=with_a)
    gbar = torch.randn((K, D), generator=torch.Generator().manual_seed(3)).to(dtype)
    if not _reduce_supported(D, dtype):
        from modelos_amd._lib import PkmError

        with pytest.raises(PkmError, match="not supported"):
            eb.eb_double_backward(*_dev(idx, a, g, gbar, device=device))
        return
    d_g, d_a = eb.eb_double_backward(*_dev(idx, a, g, gbar, device=device))
    e_g, e_a = ref.eb_double_backward(idx, a, g, gbar)
    assert_rel_close(d_g, e_g, REL_TOL[dtype], f"d_grad_output {dtype}")
    if with_a:
        assert_rel_close(d_a, e_a, REL_TOL[dtype], f"d_a {dtype}")
    else:
        assert d_a is None


def _bits_equal_fraction(a: torch.Tensor, b: torch.Tensor) -> float:
    return (a.cpu() == b.cpu()).float().mean().item()


@pytest.mark.parametrize("D", [512, 1024, 64, 4096])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
def test_backward_float32_gradient_into_half_table(dtype, D, device):
    """A float32 upstream gradient into a 16-bit table is read as float32,
    as the reference's kernel reads it (pkm/xformer_embeddingbag.py:322):
    the table gradient is the float32 sum of the unrounded products, rounded
    once, so it equals the float64 sum rounded to the table dtype except where
    that sum lies within float32 rounding of a rounding boundary (rounding the
    gradient to the table dtype first moves about a third of the entries)."""
    from modelos_amd import embedding_bag as eb

    B, L, K = 48, 32, 700
    W, idx, p, _ = eb_inputs(B, L, K, D, dtype, seed=77, psw_dtype=torch.float32, with_grad=False)
    g = torch.randn((B, D), generator=torch.Generator().manual_seed(78))
    gW, gp = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    e64W, e64p = ref.eb_backward(idx, W.double(), p.double(), g.double())
    assert gW.dtype == dtype and gp.dtype == torch.float32
    assert _bits_equal_fraction(gW, e64W.to(dtype)) > 0.999
    cW = ref.eb_backward(idx, W.double().abs(), p.double().abs(), g.double().abs())[0]
    # one rounding to the table dtype (half a unit in the last place; float16's subnormals have a
    # fixed spacing of 2^-24)
    assert_rel_close(gW, e64W, 2 ** -8 if dtype == torch.bfloat16 else 2 ** -11, "grad_weight", cond=cW,
                     atol=2 ** -25 if dtype == torch.float16 else 0.0)
    # psw-gradient: a float32 dot of the table row (exact in float32) and the float32 gradient
    cp = ref.eb_backward(idx, W.double().abs(), p.double().abs(), g.double().abs())[1]
    assert_rel_close(gp, e64p, 1e-5, "grad_psw", cond=cp)
    # the same through the fixed-scratch entry point
    from modelos_amd import _lib

    dW, didx, dp, dg = _dev(W, idx, p, g, device=device)
    gW2 = torch.empty_like(dW)
    gp2 = torch.empty_like(dp)
    _lib.call("pkm_eb_bwd_noalloc", _lib.ptr(dW), K, D, _lib.dtype_code(dW), _lib.ptr(didx), _lib.ptr(dp),
              _lib.dtype_code(dp), _lib.ptr(dg), _lib.dtype_code(dg), B, L, _lib.ptr(gW2), _lib.ptr(gp2),
              _lib.stream_of(dW.device))
    torch.cuda.synchronize()
    assert torch.equal(gW2, gW) and torch.equal(gp2, gp)


@pytest.mark.parametrize("gdt", [torch.float16, torch.bfloat16], ids=str)
def test_backward_gradient_of_other_dtype(gdt, device):
    """A 16-bit gradient into a float32 table, or a 16-bit gradient of the
    other 16-bit type: read as float32 (exact widening), so the result is the
    reference's float32 computation on those gradient values."""
    from modelos_amd import embedding_bag as eb

    B, L, K, D = 40, 16, 500, 256
    for wdt in (torch.float32, torch.bfloat16 if gdt == torch.float16 else torch.float16):
        W, idx, p, _ = eb_inputs(B, L, K, D, wdt, seed=81, psw_dtype=torch.float32, with_grad=False)
        g = torch.randn((B, D), generator=torch.Generator().manual_seed(82)).to(gdt)
        gW, gp = eb.eb_backward(*_dev(idx, W, p, g, device=device))
        e64W, e64p = ref.eb_backward(idx, W.double(), p.double(), g.double())
        assert gW.dtype == wdt
        cW = ref.eb_backward(idx, W.double().abs(), p.double().abs(), g.double().abs())[0]
        if wdt == torch.float32:
            assert_rel_close(gW, e64W, 1e-6, f"grad_weight {wdt} <- {gdt}", cond=cW)
        else:
            assert _bits_equal_fraction(gW, e64W.to(wdt)) > 0.999
        assert_rel_close(gp, e64p, 1e-5, f"grad_psw {wdt} <- {gdt}",
                         cond=ref.eb_backward(idx, W.double().abs(), p.double().abs(), g.double().abs())[1])


@pytest.mark.parametrize("gbar_dt,g_dt", [(torch.bfloat16, torch.float32), (torch.float16, torch.float32),
                                          (torch.float32, torch.bfloat16), (torch.bfloat16, torch.float16)],
                         ids=lambda v: str(v).replace("torch.", ""))
def test_double_backward_table_gradient_dtype_differs(gbar_dt, g_dt, device):
    """g_bar (the gradient of the table gradient) and the upstream gradient
    in different dtypes: g_bar [K, D] is read in its own dtype (no copy), the
    upstream gradient in its own dtype or as float32, the sums in float32
    (the reference's type promotion), d_grad_output returned in the upstream
    gradient's dtype (as autograd returns it)."""
    from modelos_amd import embedding_bag as eb

    B, L, K, D = 40, 24, 600, 256
    _, idx, a, g = eb_inputs(B, L, K, D, torch.float32, seed=79)
    g = g.to(g_dt)
    gbar = torch.randn((K, D), generator=torch.Generator().manual_seed(80)).to(gbar_dt)
    d_g, d_a = eb.eb_double_backward(*_dev(idx, a, g, gbar, device=device))
    e_g, e_a = ref.eb_double_backward(idx, a.double(), g.double(), gbar.double())
    c_g, c_a = ref.eb_double_backward(idx, a.double().abs(), g.double().abs(), gbar.double().abs())
    assert d_g.dtype == g_dt and d_a.dtype == a.dtype
    tol_g = 1e-5 if g_dt == torch.float32 else REL_TOL[g_dt]
    assert_rel_close(d_g, e_g, tol_g, "d_grad_output", cond=c_g)
    assert_rel_close(d_a, e_a, 1e-5, "d_a", cond=c_a)
    if g_dt != torch.float32:
        # the float32 sums round once: equal to the float64 result rounded to the output dtype
        assert _bits_equal_fraction(d_g, e_g.to(g_dt)) > 0.99


def test_autograd_dropin_pkm(device):
    from modelos_amd.pkm.xformer_embeddingbag import xformers_embedding_bag

    W, idx, p, g = eb_inputs(40, 32, 900, 1024, torch.bfloat16, seed=31)
    dW, didx, dp, dg = _dev(W, idx, p, g, device=device)
    dW.requires_grad_(True)
    dp.requires_grad_(True)
    out = xformers_embedding_bag(didx, dW, dp)
    out.backward(dg)
    eW, ep = ref.eb_backward(idx, W, p, g)
    assert_rel_close(out, ref.eb_forward(idx, W, p), 2e-2, "pkm drop-in forward")
    assert_rel_close(dW.grad, eW, 2e-2, "pkm drop-in weight grad")
    assert_rel_close(dp.grad, ep, 2e-2, "pkm drop-in psw grad")


@pytest.mark.parametrize("bw_algo", ["atomics", "lock"])
def test_dispatcher_bw_algo_variants(bw_algo, device):
    """xformers_embedding_bag(..., bw_algo=...) (pkm/xformer_embeddingbag.py:403-438):
    the atomics and lock variants give the reverse-indices gradients bit for
    bit (all three run the deterministic backward; the reference's "lock"
    variant returns an all-zero table gradient, a bug not reproduced), and
    match the oracle."""
    from modelos_amd.pkm.xformer_embeddingbag import xformers_embedding_bag

    W, idx, p, g = eb_inputs(64, 48, 2000, 512, torch.bfloat16, seed=37)
    idx[:, :6] = 11  # a hot row
    grads = {}
    for algo in ("reverse_indices", bw_algo):
        dW, didx, dp, dg = _dev(W, idx, p, g, device=device)
        dW.requires_grad_(True)
        dp.requires_grad_(True)
        xformers_embedding_bag(didx, dW, dp, bw_algo=algo).backward(dg)
        grads[algo] = (dW.grad.cpu(), dp.grad.cpu())
    assert torch.equal(grads[bw_algo][0], grads["reverse_indices"][0])
    assert torch.equal(grads[bw_algo][1], grads["reverse_indices"][1])
    eW, ep = ref.eb_backward(idx, W, p, g)
    assert_rel_close(grads[bw_algo][0], eW, 2e-2, f"{bw_algo} weight grad", cond=ref.eb_backward(idx, W.abs(), p.abs(), g.abs())[0])
    assert_rel_close(grads[bw_algo][1], ep, 2e-2, f"{bw_algo} psw grad")


def test_autograd_dropin_fwpkm_double_backward(device):
    """Outer gradient through one inner SGD step on the table, the fwpkm pattern
    (fwpkm/fwpkm.py:308-365): compared with the same computation done by
    autograd on the oracle's differentiable forward in float64."""
    from modelos_amd.fwpkm.xformer_embeddingbag_grad_wrapper import xformers_embedding_bag

    B, L, K, D = 24, 16, 300, 256
    W, idx, a, _ = eb_inputs(B, L, K, D, torch.float32, seed=41)
    tgt = torch.randn((B, D), generator=torch.Generator().manual_seed(42))
    idx2 = torch.randint(0, K, (B, L), generator=torch.Generator().manual_seed(43))
    a2 = torch.softmax(torch.randn((B, L), generator=torch.Generator().manual_seed(44)), -1)

    def run(eb_fn, W0, a0, dev_or_none):
        hyp = eb_fn(idx if dev_or_none is None else idx.to(dev_or_none), W0, a0)
        t = tgt if dev_or_none is None else tgt.to(dev_or_none)
        inner = 0.5 * ((hyp - t) ** 2).mean()
        (gV,) = torch.autograd.grad(inner, W0, create_graph=True)
        W1 = W0 - 0.1 * gV * (B * D)
        i2 = idx2 if dev_or_none is None else idx2.to(dev_or_none)
        p2 = a2 if dev_or_none is None else a2.to(dev_or_none)
        out = eb_fn(i2, W1, p2)
        return (out**2).sum()

    Wd = W.to(device).requires_grad_(True)
    ad = a.to(device).requires_grad_(True)
    loss = run(lambda i, w, p: xformers_embedding_bag(i, w, p), Wd, ad, device)
    gW, ga = torch.autograd.grad(loss, (Wd, ad))

    We = W.double().requires_grad_(True)
    ae = a.double().requires_grad_(True)
    loss_e = run(lambda i, w, p: ref.eb_forward(i, w, p.double()), We, ae, None)
    eW, ea = torch.autograd.grad(loss_e, (We, ae))
    assert_rel_close(loss.detach(), loss_e.detach(), 1e-5, "outer loss")
    assert_rel_close(gW, eW, 1e-5, "outer grad wrt table")
    assert_rel_close(ga, ea, 1e-5, "outer grad wrt per-sample weights")


# ---------------------------------------------------------------------------
# Full standalone size: 16384 bags x 128 lookups, 2^20 x 1024 bf16 table
# ---------------------------------------------------------------------------
@pytest.fixture(scope="module")
def full_case(device):
    B, L, K, D = 16384, 128, 1 << 20, 1024
    g = torch.Generator(device=device).manual_seed(0)
    W = (torch.randn((K, D), generator=g, device=device) * 0.03).to(torch.bfloat16)
    idx = torch.randint(0, K, (B, L), generator=g, device=device)
    p = torch.softmax(torch.randn((B, L), generator=g, device=device), -1).to(torch.bfloat16)
    gr = torch.randn((B, D), generator=g, device=device).to(torch.bfloat16)
    return W, idx, p, gr


def test_full_size_forward_sampled(full_case):
    from modelos_amd import embedding_bag as eb

    W, idx, p, _ = full_case
    out = eb.eb_forward(idx, W, p)
    sel = torch.randperm(idx.shape[0], generator=torch.Generator().manual_seed(1))[:256].to(idx.device)
    si, sp = idx[sel].cpu(), p[sel].cpu()
    rows = W[si.reshape(-1)].cpu()
    local = torch.arange(si.numel()).view(si.shape)
    expect = ref.eb_forward(local, rows, sp)
    assert_rel_close(out[sel], expect, 2e-2, "full-size forward (sampled bags)")


def test_full_size_backward_sampled_and_properties(full_case):
    from modelos_amd import embedding_bag as eb

    W, idx, p, gr = full_case
    K, D = W.shape
    gW, gp = eb.eb_backward(idx, W, p, gr)
    gW2, gp2 = eb.eb_backward(idx, W, p, gr)
    assert torch.equal(gW, gW2) and torch.equal(gp, gp2), "not bitwise deterministic"
    # untouched rows exactly zero
    touched = torch.zeros(K, dtype=torch.bool, device=idx.device)
    touched[idx.reshape(-1)] = True
    assert (gW[~touched] == 0).all()
    # checksum over all rows: sum_r gW[r] = sum_b (sum_j p[b,j]) g[b]
    colsum = gW.float().sum(0)
    expect = (p.float().sum(1, keepdim=True) * gr.float()).sum(0)
    assert_rel_close(colsum, expect, 2e-2, "column-sum checksum")
    # sampled rows against the oracle
    rows = torch.randperm(K, generator=torch.Generator().manual_seed(2))[:512].to(idx.device)
    flat = idx.reshape(-1)
    hit = torch.isin(flat, rows)
    pos = hit.nonzero().squeeze(1)
    b = pos // idx.shape[1]
    occ_rows = flat[pos]
    contrib = p.reshape(-1)[pos].float()[:, None] * gr[b].float()
    exp_rows = torch.zeros(K, D, device=idx.device).index_add_(0, occ_rows, contrib)[rows]
    assert_rel_close(gW[rows], exp_rows, 2e-2, "sampled grad_weight rows")
    # sampled psw gradients
    sb = torch.randperm(idx.shape[0], generator=torch.Generator().manual_seed(3))[:128].to(idx.device)
    e_gp = (W[idx[sb]].float() * gr[sb].float()[:, None, :]).sum(-1)
    assert_rel_close(gp[sb], e_gp, 2e-2, "sampled grad_psw")


# Upstream gradients larger than the L2 of one XCD (the g rows of every
# occurrence are re-read from the Infinity Cache): full parity at moderate
# sizes, with heavy rows, invalid indices, unweighted bags and bitwise
# determinism.
LARGE_G = [
    (4200, 16, 50000, 1024, torch.bfloat16),  # 8.6 MB of upstream gradient
    (2200, 24, 20000, 2048, torch.bfloat16),
    (2200, 8, 30000, 1024, torch.float32),
    (8800, 4, 9000, 512, torch.float16),
]


@pytest.mark.parametrize("B,L,K,D,dtype", LARGE_G, ids=lambda v: str(v).replace("torch.", ""))
def test_backward_large_gradient_parity(B, L, K, D, dtype, device):
    from modelos_amd import embedding_bag as eb

    assert B * D * torch.tensor([], dtype=dtype).element_size() > 8 << 20
    W, _, p, g = eb_inputs(B, L, K, D, dtype, seed=31 + D)
    idx = _hot_indices(B, L, K, seed=32 + D)
    gW, gp = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    eW, ep = ref.eb_backward(idx, W, p, g)
    # hot rows sum thousands of terms: elementwise against the sums of |terms|
    cW, cp = ref.eb_backward(idx, W.abs(), p.abs(), g.abs())
    assert_rel_close(gW, eW, REL_TOL[dtype], "grad_weight", cond=cW)
    assert_rel_close(gp, ep, REL_TOL[dtype], "grad_psw", cond=cp)
    assert (gp.cpu()[idx < 0] == 0).all()
    gW2, gp2 = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    assert torch.equal(gW, gW2) and torch.equal(gp, gp2)


# Hot rows of a bf16 table with 64-lane rows (at least max(257, bags / 16)
# lookups) are reduced as dense products on the matrix cores, their weights
# merged per bag. Rows in ~40% of the bags, a row held up to three times by one
# bag, a row at exactly the threshold and one just below it, a hot last row,
# a bag count that is not a multiple of the 32-bag chunk or the 128-bag tile,
# bf16 and float32 weights: elementwise against the oracle's sums of |terms|,
# and bitwise run-to-run.
def _hot_matrix_indices(B, L, K, seed):
    g = torch.Generator().manual_seed(seed)
    idx = torch.randint(20, K - 1, (B, L), generator=g)
    idx[torch.rand(B, generator=g) < 0.4, 0] = 7
    v = torch.rand(B, generator=g)
    idx[v < 0.3, 1] = 8
    idx[v < 0.1, 2] = 8
    idx[v < 0.05, 3] = 8
    hot_min = max(257, B // 16)
    bags = torch.randperm(B, generator=g)
    idx[bags[:hot_min], 4] = 9
    idx[bags[:hot_min - 1], 5] = 10
    idx[torch.rand(B, generator=g) < 0.5, 6] = K - 1
    idx[bags[-3:], 7] = -1
    return idx


@pytest.mark.parametrize("psw_dtype", [torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("B,L,K,D", [(2000, 12, 30000, 512), (1000, 16, 5000, 2048), (4100, 8, 9000, 1024),
                                     (1000, 8, 3000, 4096), (1000, 12, 3000, 4096)])
def test_backward_hot_rows_matrix_cores(B, L, K, D, psw_dtype, device):
    from modelos_amd import embedding_bag as eb

    W, _, p, g = eb_inputs(B, L, K, D, torch.bfloat16, seed=41 + D, psw_dtype=psw_dtype)
    idx = _hot_matrix_indices(B, L, K, seed=42 + D)
    gW, gp = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    eW, ep = ref.eb_backward(idx, W, p, g)
    cW, cp = ref.eb_backward(idx, W.abs(), p.abs(), g.abs())
    assert_rel_close(gW, eW, REL_TOL[torch.bfloat16], "grad_weight", cond=cW)
    assert_rel_close(gp, ep, 1e-4 if psw_dtype == torch.float32 else REL_TOL[psw_dtype], "grad_psw", cond=cp)
    assert (gp.cpu()[idx < 0] == 0).all()
    gW2, gp2 = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    assert torch.equal(gW, gW2) and torch.equal(gp, gp2)


# Unweighted bags (every weight 1) with hot rows: a bag holding a hot row k
# times merges to weight k; no psw-gradients (no dot product).
def test_backward_hot_rows_unweighted(device):
    from modelos_amd import embedding_bag as eb

    B, L, K, D = 1500, 10, 8000, 1024
    W, _, _, g = eb_inputs(B, L, K, D, torch.bfloat16, seed=63, psw=False)
    idx = _hot_matrix_indices(B, L, K, seed=64)
    gW, gp = eb.eb_backward(*_dev(idx, W, None, g, device=device))
    assert gp is None
    eW, _ = ref.eb_backward(idx, W, None, g)
    cW, _ = ref.eb_backward(idx, W.abs(), None, g.abs())
    assert_rel_close(gW, eW, REL_TOL[torch.bfloat16], "grad_weight", cond=cW)


# The merged weight of a hot row's bag is carried as bf16 hi + lo: sums that
# cancel down to the lo parts come out exact. Row 5: weight 1 + 2^-8 (float32
# weights; bf16 weights hold 1) in the even bags, -1 in the odd ones; row 6:
# held twice by the even bags (weights 1 and 2^-8, merged 1 + 2^-8), once by
# the odd ones (weight -1). Every partial sum is exact in float32, so the two
# rows' gradients are exact: 2 g (row 5: 0 for bf16 weights) and 2 g. With 12
# lookups a bag into 3000 rows the rows are hot (the matrix cores; 4 into 64 rows
# take the sparse plan's chunks), rows 5 and 6 with 32 and 48 lookups a 32-bag
# chunk, row 7 with 24: twice in every fourth bag (1 and 2^-8), once in the
# bags two after those (-1): g.
@pytest.mark.parametrize("psw_dtype", [torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("L,K,D", [(4, 64, 512), (4, 64, 1024), (12, 3000, 512), (12, 3000, 1024)])
def test_backward_hot_rows_merged_weights_exact(L, K, D, psw_dtype, device):
    from modelos_amd import embedding_bag as eb

    B = 1024
    gen = torch.Generator().manual_seed(61)
    W = (torch.randn((K, D), generator=gen) * 0.05).to(torch.bfloat16)
    idx = torch.randint(10, K, (B, L), generator=gen)
    p = torch.rand((B, L), generator=gen).to(psw_dtype)
    even = torch.arange(B) % 2 == 0
    w5 = 1 + 2.0**-8 if psw_dtype == torch.float32 else 1.0
    idx[:, 0] = 5
    p[:, 0] = torch.where(even, torch.tensor(w5), torch.tensor(-1.0)).to(psw_dtype)
    idx[:, 1] = 6
    p[:, 1] = torch.where(even, torch.tensor(1.0), torch.tensor(-1.0)).to(psw_dtype)
    idx[even, 2] = 6
    p[even, 2] = 2.0**-8
    if L > 4:
        first, other = torch.arange(B) % 4 == 0, torch.arange(B) % 4 == 2
        idx[first, 3], p[first, 3] = 7, 1.0
        idx[first, 4], p[first, 4] = 7, 2.0**-8
        idx[other, 3], p[other, 3] = 7, -1.0
    col = torch.arange(D) % 3
    g = (1.0 + col).expand(B, D).to(torch.bfloat16).contiguous()  # 1, 2, 3 in every bag
    gW, gp = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    gW = gW.cpu().float()
    want5 = (2.0 * (1.0 + col) if psw_dtype == torch.float32 else torch.zeros(D)).float()
    assert torch.equal(gW[5], want5)
    assert torch.equal(gW[6], (2.0 * (1.0 + col)).float())
    if L > 4:
        assert torch.equal(gW[7], (1.0 + col).float())
    eW, ep = ref.eb_backward(idx, W, p, g)
    cW, cp = ref.eb_backward(idx, W.abs(), p.abs(), g.abs())
    assert_rel_close(gW, eW, REL_TOL[torch.bfloat16], "grad_weight", cond=cW)
    assert_rel_close(gp, ep, 1e-4 if psw_dtype == torch.float32 else REL_TOL[psw_dtype], "grad_psw", cond=cp)


# Hot rows whose 32-bag chunks hold fewer than 32 lookups, exactly 31, 32 and
# 33, and many more (a bag holding a row up to L times: a run that spans waves),
# with bags in between that do not hold the row, and a last chunk of 28 bags.
# Tolerances as above: one bf16 rounding of sums taken in another order.
@pytest.mark.parametrize("L", [48, 200])
def test_backward_hot_rows_chunk_densities(L, device):
    from modelos_amd import embedding_bag as eb

    B, K, D = 700, 3000, 512
    W, _, p, g = eb_inputs(B, L, K, D, torch.bfloat16, seed=71 + L)
    gen = torch.Generator().manual_seed(72 + L)
    idx = torch.randint(20, K, (B, L), generator=gen)
    bag = torch.arange(B)
    idx[:, 0] = 5  # 32 a chunk
    idx[bag % 32 != 7, 1] = 6  # 31, the empty bag inside
    idx[:, 2] = 7
    idx[bag % 32 == 31, 3] = 7  # 33, the chunk's last bag twice
    idx[bag % 2 == 1, 4] = 8  # 16, every other bag
    for b in range(B):  # 0 to L - 8 lookups of row 9
        idx[b, 8:8 + (b * 37) % (L - 7)] = 9
    idx[100:130, 8:] = 9  # whole bags of one row
    gW, gp = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    eW, ep = ref.eb_backward(idx, W, p, g)
    cW, cp = ref.eb_backward(idx, W.abs(), p.abs(), g.abs())
    assert_rel_close(gW, eW, REL_TOL[torch.bfloat16], "grad_weight", cond=cW)
    assert_rel_close(gp, ep, REL_TOL[torch.bfloat16], "grad_psw", cond=cp)
    gW2, gp2 = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    assert torch.equal(gW, gW2) and torch.equal(gp, gp2)


# Hot rows with long runs of 32-bag chunks that do not hold them (written by a
# wave, shorter ones by a lane: 8 chunks and 9): before the first, between two,
# after the last; the end of one such row and the start of the next in one wave.
def test_backward_hot_rows_chunk_gaps(device):
    from modelos_amd import embedding_bag as eb

    B, L, K, D = 4100, 6, 3000, 512
    W, _, p, g = eb_inputs(B, L, K, D, torch.bfloat16, seed=91)
    idx = torch.randint(100, K, (B, L), generator=torch.Generator().manual_seed(92))
    idx[600:900, 0] = 5  # then 100 chunks without
    idx[-300:, 0] = 6
    idx[1000:1200, 0] = 7  # before, between and after
    idx[3000:3100, 0] = 7
    for c in range(0, B - 64, 9 * 32):  # every ninth chunk
        idx[c:c + 32, 1] = 8
    for c in range(0, B - 64, 10 * 32):
        idx[c:c + 32, 2] = 9
    for r in range(8):  # rows 10 to 17: 260 lookups each, 44 bags
        idx[64 * r:64 * r + 44] = 10 + r
        idx[64 * r + 43, 4:] = 20
    gW, gp = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    eW, ep = ref.eb_backward(idx, W, p, g)
    cW, cp = ref.eb_backward(idx, W.abs(), p.abs(), g.abs())
    assert_rel_close(gW, eW, REL_TOL[torch.bfloat16], "grad_weight", cond=cW)
    assert_rel_close(gp, ep, REL_TOL[torch.bfloat16], "grad_psw", cond=cp)
    gW2, gp2 = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    assert torch.equal(gW, gW2) and torch.equal(gp, gp2)


# The sparse plan's edges: the one-workgroup sort's last size and the two-level
# sort after it, the last row count it takes and one row fewer (the general
# plan), one and two keys of 8-bit digits; runs of 1 to 300 lookups across
# windows, waves and heavy chunks, a run of the first and of the last row,
# out-of-range lookups; weighted, unweighted, a float32 gradient of a 16-bit
# table. Also prepared ahead and accumulating, bit for bit.
@pytest.mark.parametrize("dtype,D", [(torch.float32, 256), (torch.float32, 2048), (torch.bfloat16, 512),
                                     (torch.bfloat16, 4096), (torch.float16, 1024), (torch.bfloat16, 64),
                                     (torch.bfloat16, 256)], ids=str)
@pytest.mark.parametrize("B,L,K", [(3, 5, 70), (80, 128, 200), (80, 128, 70000), (10241, 1, 40964), (10241, 1, 40963),
                                   (41, 301, 70001)])
def test_backward_sparse_plan(B, L, K, D, dtype, device):
    from modelos_amd import embedding_bag as eb

    W, _, p, g = eb_inputs(B, L, K, D, dtype, seed=81 + D)
    gen = torch.Generator().manual_seed(82)
    flat = torch.randint(0, K, (B * L,), generator=gen)
    pos = torch.randperm(B * L, generator=gen)
    at = 0
    for row, n in ((0, 3), (1, 16), (2, 17), (3, 64), (4, 65), (5, 256), (6, 257), (7, 300), (K - 1, 40), (-1, 5), (K, 4)):
        if at + n <= B * L // 2:
            flat[pos[at:at + n]] = row
            at += n
    idx = flat.view(B, L)
    args = _dev(idx, W, p, g, device=device)
    eW, ep = ref.eb_backward(idx, W, p, g)
    cW, cp = ref.eb_backward(idx, W.abs(), p.abs(), g.abs())
    gW, gp = eb.eb_backward(*args)
    assert_rel_close(gW, eW, REL_TOL[dtype], "grad_weight", cond=cW)
    assert_rel_close(gp, ep, REL_TOL[dtype], "grad_psw", cond=cp)
    assert (gp.cpu()[(idx < 0) | (idx >= K)] == 0).all()
    pW, pp = eb.eb_backward(*args, prepared=eb.eb_backward_prepare(args[0], args[1], args[2]))
    assert torch.equal(pW, gW) and torch.equal(pp, gp)
    pending = torch.randn((K, D), generator=gen).to(dtype).to(device)
    res = eb.eb_backward_into(*args, pending.clone())
    if res is not None:  # (64-lane rows)
        assert torch.equal(res[0], pending + gW) and torch.equal(res[1], gp)
    uW, up = eb.eb_backward(args[0], args[1], None, args[3])
    assert up is None
    assert_rel_close(uW, ref.eb_backward(idx, W, None, g)[0], REL_TOL[dtype], "unweighted",
                     cond=ref.eb_backward(idx, W.abs(), None, g.abs())[0])
    if dtype != torch.float32:
        wW, wp = eb.eb_backward(args[0], args[1], args[2], args[3].float())
        assert_rel_close(wW, eW, REL_TOL[dtype], "float32 gradient", cond=cW)
        assert_rel_close(wp, ep, REL_TOL[dtype], "float32 gradient, psw", cond=cp)


# The sparse plan with no lookup in range (both sorts): zeros everywhere, and a
# pending gradient unchanged.
@pytest.mark.parametrize("B,L,K,D,dtype", [(7, 5, 300, 512, torch.bfloat16), (7, 5, 300, 64, torch.float32),
                                           (11000, 1, 50000, 512, torch.float32)], ids=str)
def test_backward_sparse_plan_nothing_in_range(B, L, K, D, dtype, device):
    from modelos_amd import embedding_bag as eb

    W, idx, p, g = eb_inputs(B, L, K, D, dtype, seed=84)
    idx[::2], idx[1::2] = -1, K
    args = _dev(idx, W, p, g, device=device)
    gW, gp = eb.eb_backward(*args)
    assert not gW.any() and not gp.any()
    pW, pp = eb.eb_backward(*args, prepared=eb.eb_backward_prepare(args[0], args[1], args[2]))
    assert not pW.any() and not pp.any()
    pending = torch.randn((K, D), generator=torch.Generator().manual_seed(1)).to(dtype).to(device)
    res = eb.eb_backward_into(*args, pending.clone())
    if res is not None:
        assert torch.equal(res[0], pending) and not res[1].any()


# Weights of another dtype than the table's on the sparse plan, both sorts, in a
# row's lanes and in its tail (300 lookups of row 5, 200 of row 6).
@pytest.mark.parametrize("dtype,psw_dtype", [(torch.bfloat16, torch.float32), (torch.bfloat16, torch.float16),
                                             (torch.float32, torch.bfloat16)], ids=str)
@pytest.mark.parametrize("B,L,K,D", [(30, 40, 900, 1024), (30, 40, 900, 64), (400, 30, 50000, 512)])
def test_backward_sparse_plan_other_weight_dtype(B, L, K, D, dtype, psw_dtype, device):
    from modelos_amd import embedding_bag as eb

    W, idx, p, g = eb_inputs(B, L, K, D, dtype, seed=85, psw_dtype=psw_dtype)
    idx.view(-1)[:600:2] = 5
    idx.view(-1)[1:401:2] = 6
    gW, gp = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    assert gp.dtype == psw_dtype
    eW, ep = ref.eb_backward(idx, W, p, g)
    cW, cp = ref.eb_backward(idx, W.abs(), p.abs(), g.abs())
    assert_rel_close(gW, eW, REL_TOL[dtype], "grad_weight", cond=cW)
    assert_rel_close(gp, ep, REL_TOL[psw_dtype], "grad_psw", cond=cp)


# The sparse plan at a training layer's lookups: a fourth of the rows, windows of
# 16, zeros of 1 GiB beside the sort, runs across windows, a heavy row (300), rows
# of 200 and of 64, out-of-range lookups. Sampled rows against the oracle's sums,
# rows without lookups zero, prepared and direct the same bits.
def test_backward_sparse_plan_many_lookups(device):
    from modelos_amd import embedding_bag as eb

    B, L, K, D = 1024, 256, 1 << 20, 512
    gen = torch.Generator(device=device).manual_seed(86)
    W = (torch.randn((K, D), generator=gen, device=device) * D**-0.5).to(torch.bfloat16)
    idx = torch.randint(20, K, (B, L), generator=gen, device=device)
    pos = torch.randperm(B * L, generator=gen, device=device)
    at = 0
    for row, n in ((3, 300), (4, 200), (5, 64), (6, 17), (7, 16), (K - 1, 70), (-1, 9), (K, 9)):
        idx.view(-1)[pos[at:at + n]] = row
        at += n
    p = torch.softmax(torch.randn((B, L), generator=gen, device=device), -1).to(torch.bfloat16)
    g = torch.randn((B, D), generator=gen, device=device).to(torch.bfloat16)
    gW, gp = eb.eb_backward(idx, W, p, g)
    flat = idx.view(-1)
    touched = torch.zeros(K, dtype=torch.bool, device=device)
    touched[flat[(flat >= 0) & (flat < K)]] = True
    assert not gW[~touched].any()
    some = torch.randint(20, K, (400,), generator=gen, device=device)
    rows = torch.cat([torch.arange(3, 8, device=device), torch.tensor([K - 1], device=device), some[touched[some]]])
    for r in rows.tolist():
        at = (flat == r).nonzero()[:, 0]
        terms = g[at // L].double() * p.view(-1)[at, None].double()
        err = (gW[r].double() - terms.sum(0)).abs()
        assert (err <= REL_TOL[torch.bfloat16] * terms.abs().sum(0)).all(), f"row {r}"
    bags = torch.randint(0, B, (64,), generator=gen, device=device)
    j = idx[bags]
    inside = (j >= 0) & (j < K)
    terms = W[j.clamp(0, K - 1)].double() * g[bags, None].double()
    err = (gp[bags].double() - terms.sum(-1)).abs()
    assert (err[inside] <= REL_TOL[torch.bfloat16] * terms.abs().sum(-1)[inside]).all()
    assert not gp[(idx < 0) | (idx >= K)].any()
    pW, pp = eb.eb_backward(idx, W, p, g, prepared=eb.eb_backward_prepare(idx, W, p))
    assert torch.equal(pW, gW) and torch.equal(pp, gp)


# The digit counts' prefix sum (256 words a tile of 4096 lookups): one block up
# to 8192 words, three launches past it; one and two digits, and few words.
@pytest.mark.parametrize("B,L,K", [(10241, 1, 40000), (1024, 128, 60000), (131073, 1, 60000), (1024, 128, 250)])
def test_backward_digit_scan_sizes(B, L, K, device):
    from modelos_amd import embedding_bag as eb

    W, idx, p, g = eb_inputs(B, L, K, 8, torch.float32, seed=83)
    idx.view(-1)[::1001] = -1
    gW, gp = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    eW, ep = ref.eb_backward(idx, W, p, g)
    cW, cp = ref.eb_backward(idx, W.abs(), p.abs(), g.abs())
    assert_rel_close(gW, eW, REL_TOL[torch.float32], "grad_weight", cond=cW)
    assert_rel_close(gp, ep, REL_TOL[torch.float32], "grad_psw", cond=cp)


# Rows longer than the row kernel's prefetch but below the heavy threshold
# (5..250 lookups), packed into the first 64-row windows, beside two heavy rows
# and uniform rows: with more than 3 lookups per row on average (the 8-slot
# prefetch) and fewer (4 slots; 2 for float32 rows of 1024).
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("K", [2000, 40000])
def test_backward_clustered_long_rows(K, dtype, device):
    from modelos_amd import embedding_bag as eb

    B, L, D = 512, 128, 1024
    g = torch.Generator().manual_seed(61)
    counts = torch.randint(5, 251, (200,), generator=g)
    ids = [torch.full((int(c),), r) for r, c in enumerate(counts)]
    ids += [torch.full((400,), 300), torch.full((1000,), 301)]
    ids = torch.cat(ids)
    rest = torch.randint(0, K, (B * L - ids.numel(),), generator=g)
    idx = torch.cat([ids, rest])[torch.randperm(B * L, generator=g)].view(B, L)
    W, _, p, gr = eb_inputs(B, L, K, D, dtype, seed=62)
    gW, gp = eb.eb_backward(*_dev(idx, W, p, gr, device=device))
    eW, ep = ref.eb_backward(idx, W, p, gr)
    cW, cp = ref.eb_backward(idx, W.abs(), p.abs(), gr.abs())
    assert_rel_close(gW, eW, REL_TOL[dtype], "grad_weight", cond=cW)
    assert_rel_close(gp, ep, REL_TOL[dtype], "grad_psw", cond=cp)
    gW2, gp2 = eb.eb_backward(*_dev(idx, W, p, gr, device=device))
    assert torch.equal(gW, gW2) and torch.equal(gp, gp2)


# Row counts past 2^20 change the sort's digit plan: 2 passes of 11-bit digits
# up to 2^22 rows, 3 passes of 10-bit digits beyond. Indices also sit on the
# digit boundaries and at the last row.
WIDE_K = [(700, 40, 3_000_000, 16), (300, 50, 5_000_000, 8)]


@pytest.mark.parametrize("B,L,K,D", WIDE_K, ids=lambda v: str(v))
def test_backward_wide_key_range(B, L, K, D, device):
    from modelos_amd import embedding_bag as eb

    dtype = torch.float32
    W, _, p, g = eb_inputs(B, L, K, D, dtype, seed=51 + D)
    idx = _hot_indices(B, L, K, seed=52 + D)
    edge = torch.tensor([0, 1, (1 << 10) - 1, 1 << 10, (1 << 11) - 1, 1 << 11, (1 << 20) - 1, 1 << 20,
                         (1 << 21) + 5, (1 << 22) - 1, K - 2, K - 1])
    edge = edge[edge < K]
    idx.view(-1)[-3 * edge.numel():] = edge.repeat(3)
    gW, gp = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    eW, ep = ref.eb_backward(idx, W, p, g)
    cW, cp = ref.eb_backward(idx, W.abs(), p.abs(), g.abs())
    assert_rel_close(gW, eW, REL_TOL[dtype], "grad_weight", cond=cW)
    assert_rel_close(gp, ep, REL_TOL[dtype], "grad_psw", cond=cp)
    assert (gp.cpu()[idx < 0] == 0).all()


def test_backward_large_gradient_unweighted(device):
    from modelos_amd import embedding_bag as eb

    B, L, K, D = 4200, 8, 20000, 1024
    W, idx, _, g = eb_inputs(B, L, K, D, torch.bfloat16, seed=41, psw=False)
    gW, gp = eb.eb_backward(*_dev(idx, W, None, g, device=device))
    assert gp is None
    eW, _ = ref.eb_backward(idx, W, None, g)
    assert_rel_close(gW, eW, REL_TOL[torch.bfloat16], "unweighted grad_weight")


PREP_CASES = [
    (33, 17, 1000, 1024, torch.bfloat16, True),
    (9, 65, 300, 256, torch.float32, True),
    (5, 128, 2000, 2048, torch.float16, False),
    (17, 31, 100, 128, torch.bfloat16, True),
    (4, 2, 10, 32, torch.float32, True),
    (0, 8, 100, 512, torch.bfloat16, True),
    (512, 256, 70000, 1024, torch.bfloat16, True),
]


@pytest.mark.parametrize("B,L,K,D,dtype,weighted", PREP_CASES, ids=lambda v: str(v).replace("torch.", ""))
def test_backward_prepared_matches_direct(B, L, K, D, dtype, weighted, device):
    """pkm_eb_bwd_prepare on the side stream, then pkm_eb_bwd_prepared on the
    current one, gives pkm_eb_bwd's outputs bit for bit, out-of-range lookups
    (psw-gradient 0) included."""
    from modelos_amd import embedding_bag as eb

    W, idx, p, g = eb_inputs(B, L, K, D, dtype, seed=41 + B)
    if B > 2:
        idx[1, 0] = -1
        idx[2, -1] = K + 5
    dW, didx, dp, dg = _dev(W, idx, p if weighted else None, g, device=device)
    gw0, gp0 = eb.eb_backward(didx, dW, dp, dg)
    prep = eb.eb_backward_prepare(didx, dW, dp)
    gw1, gp1 = eb.eb_backward(didx, dW, dp, dg, prepared=prep)
    torch.cuda.synchronize()
    assert torch.equal(gw0, gw1)
    if weighted:
        assert torch.equal(gp0, gp1)
        if B > 2:
            assert gp1[1, 0].item() == 0.0 and gp1[2, -1].item() == 0.0
    eW, ep = ref.eb_backward(idx, W, p if weighted else None, g)
    tol = REL_TOL[dtype]
    assert_rel_close(gw1, eW, tol, "prepared weight grad", cond=ref.eb_backward(idx, W.abs(), p.abs() if weighted else None, g.abs())[0])
    if weighted:
        assert_rel_close(gp1, ep, tol, "prepared psw grad")


def test_backward_prepared_rejects_other_lookups(device):
    from modelos_amd import embedding_bag as eb

    W, idx, p, g = eb_inputs(8, 16, 500, 256, torch.bfloat16, seed=43)
    dW, didx, dp, dg = _dev(W, idx, p, g, device=device)
    prep = eb.eb_backward_prepare(didx, dW, dp)
    with pytest.raises(ValueError):
        eb.eb_backward(didx.clone(), dW, dp, dg, prepared=prep)


@pytest.mark.parametrize("K,hot", [(70000, False), (3000, False), (3000, True)])
def test_backward_prepared_workspace_serves_two_reductions(K, hot, device):
    """One prepared workspace, two reductions with different upstream
    gradients (retain_graph, or the same lookups reused): each reduction
    clears its own row-schedule counters, and leaves the hot-row lists the
    prepare built intact, so both equal pkm_eb_bwd's."""
    from modelos_amd import embedding_bag as eb

    W, idx, p, g = eb_inputs(512, 256, K, 1024, torch.bfloat16, seed=47)
    if hot:
        idx = _hot_indices(512, 256, K, seed=49)  # rows 3, 4, 5 reach the hot threshold
    g2 = (torch.randn(g.shape, generator=torch.Generator().manual_seed(48)) * 0.5).to(g.dtype)
    dW, didx, dp, dg, dg2 = _dev(W, idx, p, g, g2, device=device)
    prep = eb.eb_backward_prepare(didx, dW, dp)
    gw1, gp1 = eb.eb_backward(didx, dW, dp, dg, prepared=prep)
    gw2, gp2 = eb.eb_backward(didx, dW, dp, dg2, prepared=prep)
    ew1, ep1 = eb.eb_backward(didx, dW, dp, dg)
    ew2, ep2 = eb.eb_backward(didx, dW, dp, dg2)
    torch.cuda.synchronize()
    assert torch.equal(gw1, ew1) and torch.equal(gp1, ep1)
    assert torch.equal(gw2, ew2) and torch.equal(gp2, ep2)


def test_backward_prepared_rejects_in_place_changes(device):
    """An in-place write to indices or psw after the prepare is refused (the
    workspace holds the sorted lookups and their weights)."""
    from modelos_amd import embedding_bag as eb

    W, idx, p, g = eb_inputs(8, 16, 500, 256, torch.bfloat16, seed=44)
    dW, didx, dp, dg = _dev(W, idx, p, g, device=device)
    prep = eb.eb_backward_prepare(didx, dW, dp)
    dp.mul_(2.0)
    with pytest.raises(ValueError):
        eb.eb_backward(didx, dW, dp, dg, prepared=prep)
    prep = eb.eb_backward_prepare(didx, dW, dp)
    didx[0, 0] = 3
    with pytest.raises(ValueError):
        eb.eb_backward(didx, dW, dp, dg, prepared=prep)


# pkm_eb_bwd_accumulate: grad_weight + (the backward's table gradient), bit for
# bit the same as the backward into its own buffer followed by an add (what
# autograd forms for a table read twice), rows without lookups unchanged; on
# uniform lookups, hot rows (chunked partial sums) and clustered long rows
# (the long-row kernel). Shapes without an accumulating kernel return None.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("pattern", ["uniform", "hot", "clustered"])
def test_backward_accumulate_equals_backward_plus_add(pattern, dtype, device):
    from modelos_amd import embedding_bag as eb

    B, L, K, D = 512, 64, 40000, 1024
    W, idx, p, gr = eb_inputs(B, L, K, D, dtype, seed=71)
    if pattern == "hot":
        idx = _hot_indices(B, L, K, seed=72)
    elif pattern == "clustered":
        g = torch.Generator().manual_seed(73)
        ids = torch.cat([torch.full((int(c),), r) for r, c in enumerate(torch.randint(5, 200, (60,), generator=g))])
        rest = torch.randint(0, K, (B * L - ids.numel(),), generator=g)
        idx = torch.cat([ids, rest])[torch.randperm(B * L, generator=g)].view(B, L)
    pending = torch.randn((K, D), generator=torch.Generator().manual_seed(74)).to(dtype)
    args = _dev(idx, W, p, gr, device=device)
    gW, gp = eb.eb_backward(*args)
    want = gW + pending.to(device)
    buf = pending.to(device)
    res = eb.eb_backward_into(*args, buf)
    assert res is not None
    got, gp2 = res
    assert got.data_ptr() == buf.data_ptr()
    assert torch.equal(got, want)
    assert torch.equal(gp2, gp)
    untouched = torch.ones(K, dtype=torch.bool)
    untouched[idx[idx >= 0].unique()] = False
    assert torch.equal(got.cpu()[untouched], pending[untouched])


def test_backward_accumulate_unsupported_returns_none(device):
    from modelos_amd import embedding_bag as eb

    B, L, K = 64, 16, 3000
    W, idx, p, gr = eb_inputs(B, L, K, 64, torch.float32, seed=75)  # 16 vectors a row: no 64-lane rows
    buf = torch.zeros((K, 64), device=device)
    assert eb.eb_backward_into(*_dev(idx, W, p, gr, device=device), buf) is None
    assert torch.count_nonzero(buf) == 0
    W, idx, p, gr = eb_inputs(B, L, K, 1024, torch.bfloat16, seed=76)
    idd, Wd, pd, gd = _dev(idx, W, p, gr, device=device)
    buf = torch.zeros((K, 1024), device=device, dtype=torch.bfloat16)
    assert eb.eb_backward_into(idd, Wd, pd, gd.float(), buf) is None  # float32 gradient of a bf16 table
    assert torch.count_nonzero(buf) == 0


# Rows of more than 256 lookups on the sparse plan, whose chunks several waves
# share by columns: rows that start, end, start and end at a chunk's edge, cover
# chunks, two in one chunk, of 255 to 257 lookups, the last chunk short; 1, 2, 4
# and 8 vectors a lane, and narrow rows. Sums in chunk order: the table gradients
# are those of the same lookups with the general plan (more than 10240 lookups, the
# others out of range), bit for bit, where that uses no matrix-core products.
@pytest.mark.parametrize("dtype,D", [(torch.float32, 256), (torch.float32, 512), (torch.float32, 1024),
                                     (torch.float32, 2048), (torch.bfloat16, 4096), (torch.bfloat16, 1024),
                                     (torch.float16, 2048), (torch.bfloat16, 256), (torch.float32, 16)], ids=str)
@pytest.mark.parametrize("counts", [(256, 257, 255, 300, 212, 513, 100), (10, 246, 512, 600, 400), (1000,),
                                    (3, 257, 252, 512, 256)], ids=str)
def test_backward_sparse_plan_heavy_chunks(counts, dtype, D, device):
    from modelos_amd import embedding_bag as eb

    K, L = 700, 8
    n = sum(counts)
    B = -(-n // L)
    W, _, p, g = eb_inputs(B, L, K, D, dtype, seed=95 + n)
    gen = torch.Generator().manual_seed(96)
    flat = torch.full((B * L,), -1)
    flat[:n] = torch.cat([torch.full((c,), 5 + 3 * i) for i, c in enumerate(counts)])
    idx = flat[torch.randperm(B * L, generator=gen)].view(B, L)
    gW, gp = eb.eb_backward(*_dev(idx, W, p, g, device=device))
    eW, ep = ref.eb_backward(idx, W, p, g)
    cW, cp = ref.eb_backward(idx, W.abs(), p.abs(), g.abs())
    assert_rel_close(gW, eW, REL_TOL[dtype], "grad_weight", cond=cW)
    assert_rel_close(gp, ep, REL_TOL[dtype], "grad_psw", cond=cp)
    uW, _ = eb.eb_backward(*_dev(idx, W, None, g, device=device))  # no psw-gradients
    ones = torch.ones_like(p)
    assert torch.equal(uW, eb.eb_backward(*_dev(idx, W, ones, g, device=device))[0])
    if dtype != torch.bfloat16:
        extra = 10241 // L + 1
        idx2 = torch.cat([idx, torch.full((extra, L), -1)])
        p2, g2 = torch.cat([p, p.new_zeros((extra, L))]), torch.cat([g, g.new_zeros((extra, D))])
        big = eb.eb_backward(*_dev(idx2, W, p2, g2, device=device))
        assert torch.equal(big[0], gW)
