"""Results of the tiled products that leave through LDS, and the 256 x 256 tile's two groups of wavefronts, at the edges of tiles."""

from __future__ import annotations

import pytest
import torch

from test_gpu_kernels import _rand

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from mini_llm_runtime_amd.kernels.ops import HipOps

    return HipOps(torch.bfloat16, "cuda")


# one, two, three and seven steps of k (odd and even numbers take the two register sets in another order), tails of k; tokens and
# features around a tile, a last token tile whose second group of wavefronts has no tokens (257 .. 384)
@pytest.mark.parametrize("kernel", [23, 24, 25, 45, 46, 47, 48])
@pytest.mark.parametrize("m,n,k", [(1, 16, 8), (255, 256, 64), (257, 272, 136), (384, 528, 72), (385, 976, 200), (130, 1328, 424)])
@pytest.mark.parametrize("epilogue", ["plain", "bias", "swiglu", "geglu"])
def test_staged_results_are_the_stored_ones(ops, kernel, m, n, k, epilogue):
    """The same sums in float32 leave their own way: rounded, they are the staged bits."""
    x, w = _rand((m, k), torch.bfloat16, 71).cuda(), _rand((n, k), torch.bfloat16, 72, 0.1).cuda()
    bias = _rand((n,), torch.float32, 73).cuda() if epilogue in ("bias", "geglu") else None
    kw = {"swiglu": dict(swiglu=True), "geglu": dict(geglu=True)}.get(epilogue, {})
    staged = ops.linear(x, w, bias, mfma_kernel=kernel, **kw)
    stored = ops.linear(x, w, bias, mfma_kernel=kernel, out_dtype=torch.float32, **kw)
    assert staged.shape == stored.shape and torch.equal(staged, stored.to(torch.bfloat16))
    ref = x.double() @ w.double().t() + (0 if bias is None else bias.double())
    if not kw:  # k products of float32 accuracy, in whatever order
        bound = k * 2.0**-24 * (x.double().abs() @ w.double().abs().t()) + 2.0**-23 * ref.abs() + 1e-6
        assert ((stored.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("kernel", [23, 24, 25, 45, 46, 47, 48])
@pytest.mark.parametrize("n", [20, 100, 268])
def test_rows_of_other_widths_are_stored_directly(ops, kernel, n):
    """Rows that are no multiple of 16 bytes, and results that do not start at one."""
    x, w = _rand((140, 72), torch.bfloat16, 74).cuda(), _rand((n, 72), torch.bfloat16, 75, 0.1).cuda()
    stored = ops.linear(x, w, mfma_kernel=kernel, out_dtype=torch.float32)
    assert torch.equal(ops.linear(x, w, mfma_kernel=kernel), stored.to(torch.bfloat16))
    flat = torch.empty(140 * 256 + 4, dtype=torch.bfloat16, device="cuda")
    w = _rand((256, 72), torch.bfloat16, 76, 0.1).cuda()
    off = ops.linear(x, w, mfma_kernel=kernel, out=flat[4:].view(140, 256))
    assert torch.equal(off, ops.linear(x, w, mfma_kernel=kernel))


@pytest.mark.parametrize("kernel", [24, 25, 45])
@pytest.mark.parametrize("slices", [2, 3, 5])
def test_tiles_cut_along_k(ops, slices, kernel):
    """Slices of one, two and three steps (five steps of k in 2, 3 and 5)."""
    m, n, k = 300, 300, 264
    x, w = _rand((m, k), torch.bfloat16, 77).cuda(), _rand((n, k), torch.bfloat16, 78, 0.1).cuda()
    got = ops.linear(x, w, partial_sums=True, slices=slices, mfma_kernel=kernel)
    ref = x.double() @ w.double().t()
    bound = k * 2.0**-24 * (x.double().abs() @ w.double().abs().t()) + 1e-6
    assert got.shape == (slices, m, n) and ((got.double().sum(0) - ref).abs() <= bound).all()


# tokens in every part of a tile's rows that leave in turns, features that end inside a tile (a row of 4 n bytes is whole pieces of 16)
@pytest.mark.parametrize("kernel", [24, 25, 45, 46, 47, 48])
@pytest.mark.parametrize("m,n,k", [(1, 4, 8), (63, 132, 64), (65, 128, 200), (193, 260, 72), (257, 516, 136), (129, 324, 264)])
@pytest.mark.parametrize("slices", [1, 2])
@pytest.mark.parametrize("bias", [False, True])
def test_staged_sums_are_the_stored_ones(ops, kernel, m, n, k, slices, bias):
    """float32 sums leave through LDS where their rows start at 16 bytes; in a tensor that does not, they are stored directly."""
    x, w = _rand((m, k), torch.bfloat16, 79).cuda(), _rand((n, k), torch.bfloat16, 80, 0.1).cuda()
    b = _rand((n,), torch.float32, 81).cuda() if bias else None
    kw = dict(partial_sums=True, slices=slices) if slices > 1 else dict(out_dtype=torch.float32)
    staged = ops.linear(x, w, b, mfma_kernel=kernel, **kw)
    flat = torch.empty(staged.numel() + 1, dtype=torch.float32, device="cuda")
    stored = ops.linear(x, w, b, mfma_kernel=kernel, out=flat[1:].view(staged.shape), **kw)
    assert torch.equal(staged, stored)
    ref = x.double() @ w.double().t() + (0 if b is None else b.double())
    bound = k * 2.0**-24 * (x.double().abs() @ w.double().abs().t()) + 2.0**-23 * ref.abs() + 1e-6
    assert ((staged.double().reshape(-1, m, n).sum(0) - ref).abs() <= bound).all()


@pytest.mark.parametrize("m,n,k", [(65, 48, 64), (300, 300, 136), (1048, 3584, 3584), (2000, 2048, 2048), (2048, 3584, 7168)])
def test_sums_for_the_stream_are_not_rounded(ops, m, n, k):
    """What is added to the residual stream comes in float32 however many slices of k its product is cut into; rounded to bfloat16 the
    sums would be off by up to 2^-9 of themselves."""
    x, w = _rand((m, k), torch.bfloat16, 82).cuda(), _rand((n, k), torch.bfloat16, 83, 0.1).cuda()
    for kw in (dict(partial_sums=True), dict(for_stream=True)):
        got = ops.linear(x, w, **kw)
        assert got.dtype == torch.float32 and got.shape[1:] == (m, n)
        ref = x.double() @ w.double().t()
        bound = k * 2.0**-24 * (x.double().abs() @ w.double().abs().t()) + 2.0**-23 * ref.abs() + 1e-6
        assert ((got.double().sum(0) - ref).abs() <= bound).all()
    stream, weight = _rand((m, n), torch.float32, 84).cuda(), torch.ones(n, device="cuda")
    want = stream.double() + got.double().sum(0)
    ops.rmsnorm(stream, weight, 1e-6, delta=got)
    assert ((stream.double() - want).abs() <= 2.0**-22 * (want.abs() + got.double().abs().sum(0))).all()


# a token's factor in every part of a tile's rows; the last tile of 256 has rows for its first group of wavefronts only
@pytest.mark.parametrize("kernel", [23, 24, 25, 45, 46, 47, 48])
@pytest.mark.parametrize("m,n,k", [(130, 144, 72), (300, 272, 520)])
@pytest.mark.parametrize("way", ["rounded", "sums", "stored", "slices", "swiglu"])
def test_owed_norms(ops, kernel, m, n, k, way):
    """Rows that owe their normalisation: float32 sums times the factor, one rounding more than the sums themselves."""
    from mini_llm_runtime_amd.kernels.pending import PendingScale

    x, w = _rand((m, k), torch.bfloat16, 85, 2.0).cuda(), _rand((n, k), torch.bfloat16, 86, 0.1).cuda()
    sumsq = (torch.rand(m, 70, generator=torch.Generator().manual_seed(87)) * k * 3 / 70).cuda()
    eps = 1e-6
    owed = PendingScale(x, sumsq, torch.ones(k, dtype=torch.bfloat16).cuda(), eps, torch.zeros(m, k).cuda())
    factor = torch.rsqrt(sumsq.double().sum(1, keepdim=True) / k + eps)
    ref = factor * (x.double() @ w.double().t())
    # k roundings of the products' sum, 70 of the squares' (of which the root halves), the factor's and the last product's own
    bound = factor * (k * 2.0**-24 * (x.double().abs() @ w.double().abs().t())) + 40 * 2.0**-23 * ref.abs() + 1e-6
    if way == "swiglu":  # its 32-bit results leave from the accumulators
        got, want = (ops.linear(owed, w, swiglu=True, mfma_kernel=kernel, **kw) for kw in ({}, dict(out_dtype=torch.float32)))
        assert torch.equal(got, want.to(torch.bfloat16))
        pairs = ref.view(m, n // 4, 4)
        gate, up = pairs[..., :2].reshape(m, n // 2), pairs[..., 2:].reshape(m, n // 2)
        off = bound.view(m, n // 4, 4)
        off_gate, off_up = off[..., :2].reshape(m, n // 2), off[..., 2:].reshape(m, n // 2)
        # silu's slope is at most 1.1; its exponential and quotient are good to 2^-20
        exact = torch.nn.functional.silu(gate) * up
        assert ((want.double() - exact).abs() <= 1.1 * off_gate * (up.abs() + off_up) + gate.abs() * off_up + 2.0**-20 * exact.abs() + 1e-6).all()
        return
    kw = {"rounded": {}, "sums": dict(out_dtype=torch.float32), "slices": dict(partial_sums=True, slices=2),
          "stored": dict(out_dtype=torch.float32, out=torch.empty(m * n + 1, dtype=torch.float32, device="cuda")[1:].view(m, n))}[way]
    got = ops.linear(owed, w, mfma_kernel=kernel, **kw).double()
    if way == "slices":
        assert got.shape[0] == 2
        got = got.sum(0)
    if way == "rounded":
        bound = bound + 2.0**-8 * (ref.abs() + bound)
    assert ((got - ref).abs() <= bound).all()
