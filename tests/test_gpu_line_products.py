"""Products of up to 16 tokens by whole lines: every width of a workgroup, edges of features, steps of k and slices."""

from __future__ import annotations

import pytest
import torch

from test_gpu_kernels import _rand

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from mini_llm_runtime_amd.kernels.ops import HipOps

    return HipOps(torch.bfloat16, "cuda")


# a tail of k, one step for one wavefront, one for each, a second for some, more steps than buffers; one feature to several workgroups
@pytest.mark.parametrize("kernel", [71, 72, 73, 74])
@pytest.mark.parametrize("m", [1, 7, 16])
@pytest.mark.parametrize("n,k", [(1, 8), (20, 64), (100, 200), (64, 328), (208, 1288), (52, 4864)])
@pytest.mark.parametrize("slices", [1, 3])
def test_products(ops, kernel, m, n, k, slices):
    x, w = _rand((m, k), torch.bfloat16, 91).cuda(), _rand((n, k), torch.bfloat16, 92, 0.1).cuda()
    ref = x.double() @ w.double().t()
    bound = k * 2.0**-24 * (x.double().abs() @ w.double().abs().t()) + 1e-6
    if slices > 1:
        got = ops.linear(x, w, partial_sums=True, slices=slices, mfma_kernel=kernel).double().sum(0)
    else:
        got = ops.linear(x, w, out_dtype=torch.float32, mfma_kernel=kernel).double()
    assert got.shape == (m, n) and ((got - ref).abs() <= bound).all()


@pytest.mark.parametrize("kernel", [71, 72, 73, 74])
def test_gated_rows(ops, kernel):
    x, w = _rand((9, 264), torch.bfloat16, 93).cuda(), _rand((236, 264), torch.bfloat16, 94, 0.1).cuda()
    got, want = (ops.linear(x, w, swiglu=True, mfma_kernel=k) for k in (kernel, 11))
    # the same epilogue on sums that differ by 264 roundings at most: neighbouring bfloat16 numbers
    assert ((got.double() - want.double()).abs() <= 2.0**-7 * want.double().abs() + 1e-5).all()


# widths that make one to four blocks of 16 rows a workgroup (by the number of blocks) and leave the last workgroup some without rows
@pytest.mark.parametrize("heads,kv_heads,head_dim,hidden", [(16, 4, 128, 264), (40, 8, 64, 136), (100, 10, 48, 72), (64, 40, 128, 40), (128, 16, 128, 72)])
@pytest.mark.parametrize("tokens", [9, 16])
@pytest.mark.parametrize("rotate", [True, False])
def test_query_key_value(ops, heads, kv_heads, head_dim, hidden, tokens, rotate):
    """Against the plain product with the rotation kernel behind it, which sums in the same order and rounds at the same place."""
    width, bs = (heads + 2 * kv_heads) * head_dim, 16
    x, w = _rand((tokens, hidden), torch.bfloat16, 95).cuda(), _rand((width, hidden), torch.bfloat16, 96, 0.2).cuda()
    b = _rand((width,), torch.float32, 97).cuda()
    angles = torch.rand((tokens, head_dim // 2), generator=torch.Generator().manual_seed(98)) * 6.3
    rotation = (angles.cos().cuda(), angles.sin().cuda(), head_dim) if rotate else None
    slots = torch.arange(tokens, dtype=torch.int32, device="cuda")
    out = []
    for fused in (False, True):
        kp = torch.zeros((2, kv_heads, bs, head_dim), dtype=torch.bfloat16, device="cuda")
        vp = torch.zeros((2, kv_heads, head_dim, bs), dtype=torch.bfloat16, device="cuda")
        q = ops.qkv_rope_write(x, w, b, rotation, slots, kp, vp, num_heads=heads, num_kv_heads=kv_heads, head_dim=head_dim, block_size=bs,
                               fused=fused, mfma_kernel=16 if fused else 0)
        out.append((q[:, : heads * head_dim].float(), kp.float(), vp.float()))
    for a, c in zip(*out):  # the rotation's two products may be contracted differently: 2^-24 of either, then a last place of the result
        torch.testing.assert_close(c, a, atol=2.0**-23 * float(a.abs().amax()), rtol=2.0**-7)
