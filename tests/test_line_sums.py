"""The bound of `line_sums_room` sees what it is there to see: mistakes planted in the reference, on the CPU."""

from __future__ import annotations

import pytest
import torch

from line_sums import line_sums_room


# the longest and shortest chains that the product test has: whole lines and tiles, whole and in slices
@pytest.mark.parametrize("k,slices,lines", [(808, 1, True), (1528, 1, False), (3648, 1, True), (3648, 1, False), (2600, 2, True), (11000, 4, True),
                                            (8960, 8, True), (16384, 2, True), (22016, 8, False), (11008, 8, False)])
def test_bound_sees_rounded_slices_and_a_lost_column(k, slices, lines):
    g = torch.Generator().manual_seed(k)
    x = torch.randn((8, k), generator=g).to(torch.bfloat16)
    w = (torch.randn((64, k), generator=g) * 0.05).to(torch.bfloat16)
    b = torch.randn((64,), generator=g)
    ref, room = line_sums_room(x, w, b, slices, lines)
    cuts = [(x[:, i:j].double() @ w[:, i:j].double().t()) for i, j in zip(*(lambda e: (e[:-1], e[1:]))([k * s // slices for s in range(slices + 1)]))]
    exact = sum(cuts) + b.double()
    assert ((exact - ref).abs() <= room).all()
    rounded = sum(c.to(torch.bfloat16).double() for c in cuts) + b.double()
    assert ((rounded - ref).abs() > room).any(), "slices that are rounded to bfloat16"
    one = cuts[0].to(torch.bfloat16).double() + sum(cuts[1:]) + b.double()
    assert ((one - ref).abs() > room).any(), "one slice that is"
    lost = ref - x[:, -1:].double() @ w[:, -1:].double().t()
    assert ((lost - ref).abs() > room).any(), "the last column"
    in_order = torch.zeros(8, 64)
    for i in range(0, k, 32 if lines else 16):  # a float32 chain as long as one wavefront's would be without slices
        in_order += x[:, i : i + (32 if lines else 16)].float() @ w[:, i : i + (32 if lines else 16)].float().t()
    assert ((in_order.double() + b.double() - ref).abs() <= room).all(), "float32 sums stay inside"
