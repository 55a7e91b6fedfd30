"""The float32 kernels of the 32-bit path on the matrix cores, against float64 and against the plain kernels."""

from __future__ import annotations

import pytest
import torch

from test_gpu_kernels import _attend, _attention_reference, _paged_case, _rand
from test_gpu_prompt_attention import give_back

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from mini_llm_runtime_amd.kernels.ops import HipOps

    return HipOps(dtype=torch.float32, device="cuda:0")


def _sum_error(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """What k products and additions in float32 may be off by, in whatever order: k roundings of half a unit in the last place of
    sums that are at most the sum of the products' sizes."""
    return x.shape[1] * 2.0**-24 * (x.double().abs() @ w.double().abs().t()) + 1e-30


# edges of both kernels: one token, a full slab of 16, one more, the last of the few, the first of the tiled, a tile and one row; features around the
# 16 of a workgroup and the 64 of a tile; k of one piece, around a step of 32 and around several steps
@pytest.mark.parametrize("m", [1, 16, 17, 33, 64, 65, 129])
@pytest.mark.parametrize("n", [1, 16, 66, 130])
@pytest.mark.parametrize("k", [4, 32, 36, 100, 420])
def test_product(ops, m, n, k):
    x, w, b = _rand((m, k), torch.float32, 1), _rand((n, k), torch.float32, 2), _rand((n,), torch.float32, 3)
    ref, bound = x.double() @ w.double().t(), _sum_error(x, w)
    got = ops.linear(x.cuda(), w.cuda(), b.cuda()).cpu().double()
    assert ((got - (ref + b.double())).abs() <= bound + 2.0**-23 * (ref.abs() + b.abs())).all()


# every tiling where its last tiles hold one row or one feature (or three), k ends in a step of one piece, and the steps are odd in number (one group of
# wavefronts has one less than the other), whole and in slices of which the last is short
@pytest.mark.parametrize(
    "tiling,m,n,k,slices",
    [(221, 545, 2891, 36, 1), (221, 833, 4865, 36, 2), (211, 417, 3011, 36, 1), (211, 545, 2049, 420, 3), (212, 97, 3053, 36, 1),
     (212, 161, 1030, 420, 2), (111, 97, 4097, 36, 1), (112, 129, 33, 100, 1), (112, 97, 130, 420, 5), (112, 65, 67, 4, 1)],
)
def test_every_tiling(ops, tiling, m, n, k, slices):
    assert ops.lib.mlr_gemm_f32_tiling(m, n, k, slices) == tiling
    x, w, b = _rand((m, k), torch.float32, 16), _rand((n, k), torch.float32, 17), _rand((n,), torch.float32, 18)
    ref, bound = x.double() @ w.double().t() + b.double(), _sum_error(x, w)
    got = torch.full((slices, m, n), float("nan"), device="cuda")
    xd, wd, bd = x.cuda(), w.cuda(), b.cuda()
    ops._call(
        "mlr_gemm_f32", ops._ptr(xd), ops._ptr(wd), ops._ptr(bd), ops._ptr(got), 0, slices, m, n, k, None, None, 0.0, 0.0, ops._stream()
    )
    got = got.cpu().double().sum(0)
    assert ((got - ref).abs() <= bound + 2.0**-23 * (ref.abs() + b.abs().double())).all()


# 64 x 32 tiles up to six to a compute unit and beyond seven, 64 x 64 between; in slices of k as before
@pytest.mark.parametrize(
    "m,n,k,slices,tiling", [(480, 6528, 800, 1, 211), (325, 9511, 1360, 1, 221), (1120, 3264, 1540, 1, 221), (218, 16503, 800, 1, 211), (545, 2049, 420, 3, 211)]
)
def test_tiling_of_a_round_that_begins_late(ops, m, n, k, slices, tiling):
    assert ops.lib.mlr_gemm_f32_tiling(m, n, k, slices) == tiling


@pytest.mark.parametrize("m", [5, 40, 70])
@pytest.mark.parametrize("epilogue", ["swiglu", "clamped", "geglu", "relu2", "sigmoid", "gelu_tanh", "multiply", "rows"])
def test_epilogues_are_the_plain_kernels(ops, m, epilogue):
    n, k = 72, 64
    x, w, b = _rand((m, k), torch.float32, 4).cuda(), _rand((n, k), torch.float32, 5, 0.3).cuda(), _rand((n,), torch.float32, 6).cuda()
    kw, bias = {
        "swiglu": (dict(swiglu=True), None), "clamped": (dict(clamped_glu=(1.5, 1.7)), b), "geglu": (dict(geglu=True), b),
        "multiply": (dict(activation="sigmoid", multiply=_rand((m, n), torch.float32, 7).cuda()), b),
        "rows": (dict(multiply=_rand((9, n), torch.float32, 8).cuda(), multiply_rows=(torch.arange(m, dtype=torch.int32) % 9).cuda()), None),
    }.get(epilogue, (dict(activation=epilogue), b))
    got, plain = ops.linear(x, w, bias, **kw), ops.linear(x, w, bias, kernel="fma", **kw)
    assert got.shape == plain.shape
    # the sums differ by their order (64 roundings of values of a few units); the gatings multiply two of them
    torch.testing.assert_close(got, plain, atol=2e-4, rtol=2e-5)


def test_partial_sums_add_up(ops):
    x, w, b = _rand((100, 4864), torch.float32, 9), _rand((90, 4864), torch.float32, 10), _rand((90,), torch.float32, 11)
    got = ops.linear(x.cuda(), w.cuda(), b.cuda(), partial_sums=True).cpu().double()
    assert got.dim() == 3 and got.shape[1:] == (100, 90)
    ref = x.double() @ w.double().t() + b.double()
    assert ((got.sum(0) - ref).abs() <= _sum_error(x, w) + 2.0**-23 * ref.abs()).all()


def test_operands_off_16_bytes_take_the_plain_kernel(ops):
    """A view that starts 4 bytes into a tensor is no operand for 16-byte loads: same result, another kernel."""
    flat = _rand((64 * 70 + 1,), torch.float32, 12).cuda()
    x, w = flat[1:].view(70, 64), _rand((32, 64), torch.float32, 13).cuda()
    torch.testing.assert_close(ops.linear(x, w), ops.linear(x, w, kernel="fma"), atol=0, rtol=0)
    torch.testing.assert_close(ops.linear(x, w), ops.linear(x.clone(), w), atol=1e-4, rtol=1e-5)


@pytest.mark.parametrize("heads,kv_heads,head_dim,block", [(14, 2, 64, 16), (4, 4, 16, 4), (3, 1, 80, 8), (6, 2, 96, 32), (4, 1, 128, 16), (2, 1, 48, 12), (2, 2, 32, 128)])
@pytest.mark.parametrize("mask", [dict(window=None), dict(window=37), dict(window=None, chunk=50)])
def test_prompt_attention(ops, heads, kv_heads, head_dim, block, mask):
    """Whole prompts around the tile's 64 queries, portions behind cached tokens, single tokens beside them."""
    entries = [(64, 64), (65, 65), (2, 2), (200, 1), (131, 131), (150, 33), (1, 1)]
    q, kp, vp, table, ctx, dense, te, pos = _paged_case(entries, heads, kv_heads, head_dim, block, torch.float32, 14)
    args = (q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx)
    sinks = _rand((heads,), torch.float32, 15).cuda()
    kw = dict(num_heads=heads, num_kv_heads=kv_heads, head_dim=head_dim, block_size=block, scale=head_dim**-0.5, **mask)
    for sink in (None, sinks):
        got = _attend(ops, *args, sinks=sink, **kw).cpu()
        plain = _attend(ops, *args, kernel="fma", sinks=sink, **kw).cpu()
        # weights add up to one and values are a few units: sums of 64 to 200 products in another order
        torch.testing.assert_close(got, plain, atol=5e-6, rtol=1e-5)
    if "chunk" not in mask:
        ref = _attention_reference(q, dense, te, pos, heads, kv_heads, head_dim, head_dim**-0.5, mask["window"])
        torch.testing.assert_close(_attend(ops, *args, **kw).cpu().double(), ref, atol=5e-6, rtol=1e-5)


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("window", [None, 70, 300])
def test_prompt_attention_over_several_turns(ops, head_dim, window):
    """Key tiles for one group of wavefronts and for both, an odd and an even number of them, several turns of each; the first key visible in either's tile."""
    entries = [(321, 321), (449, 60), (128, 128), (129, 129), (32, 32), (33, 33)]
    q, kp, vp, table, ctx, dense, te, pos = _paged_case(entries, 3, 1, head_dim, 16, torch.float32, 14)
    got = _attend(ops, q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx, num_heads=3, num_kv_heads=1, head_dim=head_dim, block_size=16,
                  scale=head_dim**-0.5, window=window)
    ref = _attention_reference(q, dense, te, pos, 3, 1, head_dim, head_dim**-0.5, window)
    torch.testing.assert_close(got.cpu().double(), ref, atol=5e-6, rtol=1e-5)  # as above


@pytest.mark.parametrize("head_dim", [16, 64, 80, 96, 128])
@pytest.mark.parametrize("mask", [dict(window=None), dict(window=70), dict(window=None, chunk=96)])
@pytest.mark.parametrize("odd", [False, True])
def test_prompt_attention_by_one_group_of_wavefronts(ops, head_dim, mask, odd):
    """More workgroups than places for two groups each: one group takes a tile's keys, one tile of them, several, and behind cached tokens; a value that is not
    finite in one prompt.  A step whose longest prompt is known to be long keeps two groups up to head size 64: the same in another order."""
    entries = [(64, 64), (65, 65), (3, 3), (150, 33), (130, 130), (200, 90), (128, 128)]
    q, kp, vp, table, ctx, *_ = _paged_case(entries, 48, 8, head_dim, 16, torch.float32, 19)
    if odd:
        vp[table[4, 100 // 16], 1, 5, 100 % 16] = float("inf")
    tiles, groups = ctx.num_query_tiles, ops.attention_library(head_dim).mlr_attention_prefill_f32_groups
    assert tiles * 48 > 512 and groups(tiles, 0, 48, mask["window"] or 0, mask.get("chunk", 0)) == 1
    args = (q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx)
    kw = dict(num_heads=48, num_kv_heads=8, head_dim=head_dim, block_size=16, scale=head_dim**-0.5, sinks=_rand((48,), torch.float32, 15).cuda(), **mask)
    got, plain = _attend(ops, *args, **kw).cpu(), _attend(ops, *args, kernel="fma", **kw).cpu()
    assert torch.isfinite(plain).all() != odd
    torch.testing.assert_close(got, plain, atol=5e-6, rtol=1e-5, equal_nan=True)
    ctx.longest_prompt_tiles = 8
    torch.testing.assert_close(_attend(ops, *args, **kw).cpu(), plain, atol=5e-6, rtol=1e-5, equal_nan=True)


@pytest.mark.parametrize("head_dim,block", [(64, 16), (128, 16), (80, 8), (16, 4)])
@pytest.mark.parametrize("mask", [dict(window=None), dict(window=20), dict(window=None, chunk=24)])
@pytest.mark.parametrize("odd", [float("nan"), float("inf")])
def test_values_that_are_not_finite_stay_with_the_tokens_that_see_them(ops, head_dim, block, mask, odd):
    """0 * inf is NaN: a value that a token does not see must not enter its sum at all, as in the plain kernel."""
    entries = [(130, 130), (190, 61)]
    q, kp, vp, table, ctx, *_ = _paged_case(entries, 2, 1, head_dim, block, torch.float32, 17)
    for entry, p in ((0, 70), (0, 129), (1, 131), (1, 150)):
        vp[table[entry, p // block], 0, 3, p % block] = odd
    vp[table[0, 10 // block], 0, :, 10 % block] = -odd
    args = (q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx)
    kw = dict(num_heads=2, num_kv_heads=1, head_dim=head_dim, block_size=block, scale=head_dim**-0.5, **mask)
    got, plain = _attend(ops, *args, **kw).cpu(), _attend(ops, *args, kernel="fma", **kw).cpu()
    assert torch.isfinite(plain[:10]).all() and not torch.isfinite(plain[129]).all()
    torch.testing.assert_close(got, plain, atol=5e-6, rtol=1e-5, equal_nan=True)


def test_prompt_attention_refuses_a_page_that_is_not_there(ops):
    q, kp, vp, table, ctx, *_ = _paged_case([(100, 100), (70, 70)], 2, 1, 64, 16, torch.float32, 16)
    table = table.clone()
    table[1, 2] = kp.shape[0]  # a visible page of the second request
    kw = dict(num_heads=2, num_kv_heads=1, head_dim=64, block_size=16, scale=0.125, window=None)
    got = _attend(ops, q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx, **kw).cpu()
    assert torch.isfinite(got[:100]).all() and torch.isnan(got[100 + 64 :]).all()


@pytest.mark.parametrize("mask", [dict(window=None), dict(window=20), dict(window=None, chunk=24)])
@pytest.mark.parametrize("page", [-1, 10**6])
def test_a_page_that_is_not_there_concerns_the_tokens_that_see_it(ops, mask, page):
    """Those rows and no others are NaN, as in the plain kernel."""
    q, kp, vp, table, ctx, *_ = _paged_case([(100, 100), (190, 70)], 2, 1, 64, 16, torch.float32, 16)
    table = table.clone()
    table[0, 2] = table[1, 8] = page  # positions 32..47 of the first request, 128..143 of the second
    args = (q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx)
    kw = dict(num_heads=2, num_kv_heads=1, head_dim=64, block_size=16, scale=0.125, **mask)
    got, plain = _attend(ops, *args, **kw).cpu(), _attend(ops, *args, kernel="fma", **kw).cpu()
    assert torch.isfinite(plain[:32]).all() and torch.isnan(plain[40]).all() and torch.isfinite(plain[100:108]).all()
    torch.testing.assert_close(got, plain, atol=5e-6, rtol=1e-5, equal_nan=True)


@pytest.mark.parametrize("head_dim,block", [(64, 16), (128, 32), (16, 4), (48, 12)])
@pytest.mark.parametrize("mask", [dict(window=1), dict(window=17), dict(window=65), dict(window=None, chunk=48), dict(window=None, chunk=160)])
def test_pages_that_were_given_back(ops, head_dim, block, mask):
    entries = [(200, 70), (331, 5), (192, 130), (448, 64), (403, 140), (300, 1)]
    q, kp, vp, table, ctx, *_ = _paged_case(entries, 2, 1, head_dim, block, torch.float32, 18)
    kw = dict(num_heads=2, num_kv_heads=1, head_dim=head_dim, block_size=block, scale=head_dim**-0.5, **mask)
    whole = _attend(ops, q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx, **kw).cpu()
    left = give_back(entries, kp, vp, table, block, **mask)
    got = _attend(ops, q.cuda(), *(t.cuda() for t in left), ctx, **kw).cpu()
    assert torch.isfinite(whole).all() and torch.equal(got, whole)
