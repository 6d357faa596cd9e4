"""The streaming scoring kernel against the oracle (GPU).

pkm_score_topk sends bfloat16 dot scores with knn <= 32 and a half key dim
of 128 or 256 (the layer's configuration) to its streaming kernel, which keeps
a sorted running top-32 per token in registers and appends the scores that
can reach it to LDS slots, merging 32 at a time. The cases aim at its own
paths: workgroup and wave tails (token counts that are not multiples of 256
or 64), head counts whose 2H does not divide the 8 XCDs, every knn up to 32,
the largest n_keys, all-equal scores (a zero query: index order), key orders
in which every score beats all earlier ones (every tile appends all of its
scores, so the wave merges after every tile) or none does, +0 / -0 ties, and
many tokens at the layer's shape.
"""
from __future__ import annotations

import pytest
import torch

from modelos_amd.product_keys import score_topk
from oracle import pkm as ref
from tests.helpers import REL_TOL, assert_rel_close, gen

pytestmark = pytest.mark.gpu

# (tokens, heads, n_keys, half, knn)
INT_SHAPES = [
    (1, 1, 64, 128, 1),
    (63, 3, 192, 128, 7),
    (257, 2, 2048, 128, 32),
    (300, 8, 1024, 256, 32),
    (65, 5, 512, 256, 16),
    (129, 4, 256, 256, 31),
]


def _ids(shape):
    return "N{}-H{}-n{}-h{}-k{}".format(*shape)


def _run(q, k, H, knn, device):
    out = score_topk(q.to(device), k.to(device), H, knn, "dot", sub_outputs=True)
    torch.cuda.synchronize()
    return [t.cpu() for t in out]


def _check_exact(q, k, H, knn, device):
    N = q.shape[0]
    scores, idx, i1, i2, s1, s2 = _run(q, k, H, knn, device)
    e_scores, e_idx, e_i1, e_i2, e_s1, e_s2 = ref.get_indices(q, k, H, knn)
    assert torch.equal(s1, e_s1) and torch.equal(s2, e_s2)
    assert torch.equal(i1, e_i1) and torch.equal(i2, e_i2)
    assert torch.equal(idx.view(N, H, knn), e_idx)
    assert torch.equal(scores.view(N, H, knn), e_scores)
    # without the sub-score outputs: the same selection
    two = score_topk(q.to(device), k.to(device), H, knn, "dot")
    assert torch.equal(two[0].cpu(), scores) and torch.equal(two[1].cpu(), idx)
    return i1


@pytest.mark.parametrize("shape", INT_SHAPES, ids=_ids)
def test_integer_inputs_bit_exact(device, shape):
    N, H, n, half, knn = shape
    g = gen(31)
    q = torch.randint(-1, 2, (N, H, 2 * half), generator=g).to(torch.bfloat16)
    k = torch.randint(-2, 3, (2 * H * n, half), generator=g).to(torch.bfloat16)
    _check_exact(q, k, H, knn, device)


@pytest.mark.parametrize("knn", list(range(1, 33)))
def test_every_knn(device, knn):
    N, H, n, half = 70, 2, 320, 128
    g = gen(100 + knn)
    q = torch.randint(-1, 2, (N, H, 2 * half), generator=g).to(torch.bfloat16)
    k = torch.randint(-2, 3, (2 * H * n, half), generator=g).to(torch.bfloat16)
    _check_exact(q, k, H, knn, device)


@pytest.mark.parametrize("shape", [(1000, 8, 1024, 256, 32), (517, 4, 512, 128, 16)], ids=_ids)
def test_random_inputs(device, shape):
    N, H, n, half, knn = shape
    g = gen(37)
    q = torch.randn((N, H, 2 * half), generator=g).to(torch.bfloat16)
    k = ((torch.rand((2 * H * n, half), generator=g) * 2 - 1) * half**-0.5).to(torch.bfloat16)
    scores, idx, i1, i2, s1, s2 = _run(q, k, H, knn, device)
    e_s1, e_s2 = ref.sub_scores(q, k, H)
    assert_rel_close(s1, e_s1, REL_TOL[torch.bfloat16], "s1")
    assert_rel_close(s2, e_s2, REL_TOL[torch.bfloat16], "s2")
    # the selection is a function of the rounded sub-scores: bit-exact
    e_scores, e_idx, e_i1, e_i2 = ref.select(s1, s2, knn)
    assert torch.equal(i1, e_i1) and torch.equal(i2, e_i2)
    assert torch.equal(idx.view(N, H, knn), e_idx)
    assert torch.equal(scores.view(N, H, knn), e_scores)


def test_zero_query_index_order(device):
    """Every score equal: the lists are the index order."""
    N, H, n, half, knn = 80, 2, 1024, 256, 32
    g = gen(41)
    q = torch.zeros((N, H, 2 * half), dtype=torch.bfloat16)
    k = torch.randn((2 * H * n, half), generator=g).to(torch.bfloat16)
    i1 = _check_exact(q, k, H, knn, device)
    assert torch.equal(i1[0, 0], torch.arange(knn))


def _one_hot_keys(N, H, n, half, col_values, seed):
    """One-hot queries (a single 1.0 per half, in column `col`) against keys
    whose column `col` holds col_values[i] for key i: every score is that
    bf16 value, exactly."""
    g = gen(seed)
    cols = torch.randint(0, half, (N, H, 2), generator=g)
    q = torch.zeros((N, H, 2, half))
    q.scatter_(3, cols[..., None], 1.0)
    K = torch.randn((H, 2, n, half), generator=g)
    for h in range(H):
        for c in range(2):
            for col in cols[:, h, c].unique().tolist():
                K[h, c, :, col] = col_values
    return q.reshape(N, H, 2 * half).to(torch.bfloat16), K.reshape(2 * H * n, half).to(torch.bfloat16)


@pytest.mark.parametrize("order", ["increasing", "decreasing", "increasing_negative"])
def test_monotone_key_orders(device, order):
    """Increasing: every tile beats everything before it (all its scores are
    appended and merged); decreasing: nothing after the first tiles passes.
    The bf16 values repeat in runs (i / 16 rounded), so ties cross tiles."""
    N, H, n, half, knn = 96, 2, 1024, 256, 32
    v = (torch.arange(n, dtype=torch.float32) + 1) / 16
    vals = {"increasing": v, "decreasing": v.flip(0), "increasing_negative": -v.flip(0)}[order]
    q, k = _one_hot_keys(N, H, n, half, vals, seed=43)
    _check_exact(q, k, H, knn, device)


def test_signed_zero_ties(device):
    """+0 and -0 scores are equal values: after the positive ones, the zeros
    come in index order whatever their sign."""
    N, H, n, half, knn = 64, 2, 256, 128, 32
    vals = torch.zeros(n)
    vals[1::2] = -0.0
    vals[torch.tensor([5, 77, 130, 200, 201, 255])] = 1.0
    vals[torch.tensor([3, 9, 100])] = -1.0
    q, k = _one_hot_keys(N, H, n, half, vals, seed=47)
    i1 = _check_exact(q, k, H, knn, device)
    zeros = [i for i in range(n) if vals[i] == 0][: knn - 6]
    assert i1[0, 0].tolist() == [5, 77, 130, 200, 201, 255] + zeros


@pytest.mark.parametrize("which", [1, 2])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
def test_single_sub_score_output_through_c_abi(device, which, dtype):
    """One sub-score pointer NULL, the other given, straight through the C ABI
    (the streaming kernel for bf16, the tile kernel for float32): the given
    half equals the full call's and the call does not touch the NULL one."""
    from modelos_amd import _lib

    N, H, n, half, knn = 300, 4, 512, 128, 32
    g = gen(77 + which)
    q = torch.randn((N, H, 2 * half), generator=g).to(dtype).to(device)
    k = torch.randn((2 * H * n, half), generator=g).to(dtype).to(device)
    full = score_topk(q, k, H, knn, "dot", sub_outputs=True)
    scores = torch.empty((N * H, knn), dtype=dtype, device=device)
    idx = torch.empty((N * H, knn), dtype=torch.long, device=device)
    s_out = torch.empty((N, H, n), dtype=dtype, device=device)
    s1, s2 = (s_out, None) if which == 1 else (None, s_out)
    _lib.call(
        "pkm_score_topk",
        _lib.ptr(q), _lib.ptr(k), N, H, n, half, knn, _lib.SCORE_CODES["dot"], _lib.dtype_code(q),
        _lib.ptr(scores), _lib.ptr(idx), None, None, _lib.ptr(s1), _lib.ptr(s2), _lib.stream_of(q.device),
    )
    torch.cuda.synchronize()
    assert torch.equal(idx, full[1]) and torch.equal(scores, full[0])
    assert torch.equal(s_out, full[4] if which == 1 else full[5])


def _repeat_tokens(q, tokens):
    return q.repeat((tokens + q.shape[0] - 1) // q.shape[0], 1, 1)[:tokens].contiguous()


# Few tokens run on the tile kernel (the smallest tile whose workgroups fit the
# chip in one round), many on the streaming one: each token's outputs are the
# same bits on both, for the streaming kernel's own cases too (the others of
# this file have few tokens). 4100 and 4353 tokens of 2 heads are past the
# tile kernel's rule, 1, 16, 17, 1025 and 2049 take its 16-, 32- and 64-token tiles.
@pytest.mark.parametrize("knn", [1, 7, 16, 31, 32])
@pytest.mark.parametrize("case", ["random", "zero", "increasing", "decreasing", "increasing_negative", "signed_zero"])
def test_few_and_many_tokens_agree(device, case, knn):
    H, n, half = 2, 1024 if case in ("increasing", "decreasing") else 512, 128 if case == "signed_zero" else 256
    N = 97
    v = (torch.arange(n, dtype=torch.float32) + 1) / 16
    g = gen(200 + knn)
    if case in ("random", "zero"):
        q = torch.randn((N, H, 2 * half), generator=g).to(torch.bfloat16)
        k = (torch.randn((2 * H * n, half), generator=g) * half**-0.5).to(torch.bfloat16)
        if case == "zero":
            q.zero_()
    else:
        vals = {"increasing": v, "decreasing": v.flip(0), "increasing_negative": -v.flip(0)}.get(case)
        if vals is None:
            vals = torch.zeros(n)
            vals[1::2] = -0.0
            vals[::97] = 1.0
        q, k = _one_hot_keys(N, H, n, half, vals, seed=201)
    many = _run(_repeat_tokens(q, 4353), k, H, knn, device)
    for tokens in (1, 16, 17, 1025, 2049, 4100):
        few = _run(_repeat_tokens(q, tokens), k, H, knn, device)
        for a, b in zip(few, many):
            assert torch.equal(a, b[: a.shape[0]]), f"{case} knn {knn} tokens {tokens}"


# Few keys: tiles of at most n / 8 tokens, the streaming kernel past the tokens
# that those hold (2 heads: 16-token tiles up to 1024 tokens of 128 keys,
# 32-token ones up to 2048 of 256 keys).
@pytest.mark.parametrize("n,knn,edge", [(64, 4, 1), (128, 8, 1024), (256, 16, 2048), (320, 16, 2048)])
def test_few_tokens_few_keys_agree(device, n, knn, edge):
    H, half = 2, 128
    g = gen(400 + n)
    q = torch.randn((89, H, 2 * half), generator=g).to(torch.bfloat16)
    k = (torch.randn((2 * H * n, half), generator=g) * half**-0.5).to(torch.bfloat16)
    many = _run(_repeat_tokens(q, 4353), k, H, knn, device)
    for tokens in (1, edge, edge + 1, 4096):
        few = _run(_repeat_tokens(q, tokens), k, H, knn, device)
        for a, b in zip(few, many):
            assert torch.equal(a, b[: a.shape[0]]), f"tokens {tokens}"


# The rule's other routes: more lanes per row in the cartesian step up to 8192
# rows, smaller tiles of float32 and of key dims the streaming kernel does not
# take, dead rows of a tile (their equal scores select nothing).
@pytest.mark.parametrize("dtype,score,half,knn", [(torch.float32, "idw", 128, 16), (torch.float32, "dot", 64, 33),
                                                  (torch.bfloat16, "dot", 64, 24), (torch.bfloat16, "idw", 128, 32),
                                                  (torch.bfloat16, "dot", 256, 64)], ids=str)
def test_few_token_tiles_agree(device, dtype, score, half, knn):
    H, n, N = 3, 1024, 6001
    g = gen(300 + knn)
    q = (torch.randn((N, H, 2 * half), generator=g) * half**-0.5).to(dtype)
    k = (torch.randn((2 * H * n, half), generator=g) * half**-0.5).to(dtype)
    many = score_topk(q.to(device), k.to(device), H, knn, score, sub_outputs=True)
    for tokens in (1, 5, 33, 700, 1400, 2700):
        few = score_topk(q[:tokens].to(device), k.to(device), H, knn, score, sub_outputs=True)
        for a, b in zip(few, many):
            assert torch.equal(a, b[: a.shape[0]]), f"tokens {tokens}"


def test_more_rows_than_a_grid_of_wide_cartesian_rows(device):
    """2^28 + 3 rows of knn 33: 16 lanes a row in the cartesian step would be
    more threads than a grid holds, so 8 take it. The same 97 tokens over and
    over, whose outputs a short call gives."""
    if torch.cuda.mem_get_info(device)[0] < 190 << 30:
        pytest.skip("needs 190 GiB of device memory")
    T, n, half, knn = (1 << 28) + 3, 64, 32, 33
    g = gen(500)
    few = torch.randn((97, 1, 2 * half), generator=g).to(torch.bfloat16).to(device)
    k = (torch.randn((2 * n, half), generator=g) * half**-0.5).to(torch.bfloat16).to(device)
    s0, i0 = score_topk(few, k, 1, knn, "dot")[:2]
    q = few.repeat((T + 96) // 97, 1, 1)[:T]
    scores, idx = score_topk(q, k, 1, knn, "dot")[:2]
    del q
    step = 97 << 17
    s0, i0 = s0.repeat(step // 97, 1), i0.repeat(step // 97, 1)
    for a in range(0, T, step):
        m = min(step, T - a)
        assert torch.equal(scores[a:a + m], s0[:m]) and torch.equal(idx[a:a + m], i0[:m]), f"rows from {a}"
    del scores, idx, s0, i0
    torch.cuda.empty_cache()
