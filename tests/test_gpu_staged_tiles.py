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
    """The same sums in float32 take the way without staging: rounded, they are the staged bits."""
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
