"""Routing from registers and from partial sums, and the grouped products at the edges of their tiles."""

from __future__ import annotations

import pytest
import torch

from test_gpu_kernels import _rand

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from mini_llm_runtime_amd.kernels.ops import HipOps

    return HipOps(torch.bfloat16, "cuda")


def _route(z, correction, top, groups, keep, scale, scores, normalise):
    """The rule in 64 bits; logits that are equal stay equal, and of equal choices the lowest index wins."""
    z = z.double()
    s = {"sigmoid": torch.sigmoid(z), "softmax": torch.softmax(z, -1), "chosen_softmax": z}[scores]
    c = s if correction is None else s + correction.double()
    if keep < groups:
        blocks = c.view(len(z), groups, -1)
        best = blocks.topk(min(2, blocks.shape[-1]), dim=-1).values.sum(-1)
        kept = torch.sort(best, dim=-1, descending=True, stable=True).indices[:, :keep]
        mask = torch.ones_like(best, dtype=torch.bool).scatter_(1, kept, False)
        c = blocks.masked_fill(mask[:, :, None], float("-inf")).reshape(z.shape)
    ids = torch.sort(c, dim=-1, descending=True, stable=True).indices[:, :top]
    w = s.gather(1, ids)
    if scores == "chosen_softmax":
        w = torch.softmax(w, -1)
    elif normalise:
        w = w / (w.sum(-1, keepdim=True) + 1e-20)
    return ids, w * scale


# one lane, a full wavefront, one expert more, all four registers of a lane, the most that fit; 257 experts and 80 groups: the plain kernel
@pytest.mark.parametrize("experts,top,groups,keep", [
    (1, 1, 1, 1), (5, 5, 1, 1), (64, 6, 8, 3), (64, 64, 1, 1), (65, 4, 5, 2), (192, 8, 64, 7), (256, 64, 16, 9), (257, 6, 1, 1), (160, 3, 80, 5),
])
@pytest.mark.parametrize("scores,normalise", [("sigmoid", False), ("softmax", True), ("chosen_softmax", False)])
@pytest.mark.parametrize("slices", [1, 2, 9])
def test_routing(ops, experts, top, groups, keep, scores, normalise, slices):
    tokens = 37
    # multiples of 1/16: scores are equal or further apart than rounding; one pair of equals in every row, and those cut off at 8
    g = torch.Generator().manual_seed(experts + top)
    z = torch.stack([torch.randperm(experts, generator=g) for _ in range(tokens)]).float().sub(experts // 2) / 16
    z = z.clamp(-8, 8) if scores != "chosen_softmax" else z
    if experts > 3:
        z[:, 3] = z[:, 0]
    parts = torch.stack([z / 2] + [torch.zeros_like(z)] * (slices - 2) + [z / 2]) if slices > 1 else z  # exact in any order
    want_ids, want = _route(z, None, top, groups, keep, 1.7, scores, normalise)
    ids, w = ops.route_experts(parts.cuda(), None, top=top, groups=groups, keep_groups=keep, scale=1.7, scores=scores, normalise=normalise)
    assert torch.equal(ids.cpu().long(), want_ids)
    # exp, a division and sums of at most 256 terms in float32, each within a few units of 2^-24
    assert ((w.cpu().double() - want).abs() <= (experts + 16) * 2.0**-24 * want + 1e-12).all()


# one token, a full workgroup and one token more (two kernels); every expert with matrices, all but some, one; more choices than a tile's rows
@pytest.mark.parametrize("tokens", [1, 3, 8, 9])
@pytest.mark.parametrize("routed,experts,top,groups,keep", [(64, 64, 6, 8, 4), (65, 60, 4, 5, 2), (256, 256, 64, 16, 9), (5, 1, 5, 1, 1), (40, 33, 2, 1, 1)])
def test_routing_that_sorts(ops, tokens, routed, experts, top, groups, keep):
    z, correction = _rand((tokens, routed), torch.float32, routed).cuda(), _rand((routed,), torch.float32, 3, 0.1).cuda()
    rule = dict(top=top, groups=groups, keep_groups=keep, scale=1.7)
    want_ids, want = ops.route_experts(z, correction, **rule)
    ids, w, order = ops.route_experts(z, correction, order=experts, **rule)
    assert torch.equal(ids, want_ids) and torch.equal(w, want)
    assert (order is None) == (tokens > 8)
    if order is None:
        return
    by_expert, offsets, tiles, most = (t.cpu() if isinstance(t, torch.Tensor) else t for t in order)
    pairs = want_ids.cpu().flatten()
    used = []
    for e in range(experts):
        rows = by_expert[offsets[e] : offsets[e + 1]].tolist()
        assert sorted(rows) == (pairs == e).nonzero().flatten().tolist()
        used += [[e, int(offsets[e]) + i] for i in range(0, len(rows), 16)]
    assert tiles.view(-1, 2).tolist() == used + [[-1, len(used)]] * (most - len(used))


# pairs around a workgroup's threads and what its registers hold, experts around what its memory holds; ids without matrices among them
@pytest.mark.parametrize("experts,pairs", [(1, 1), (64, 1023), (3, 1025), (64, 4096), (60, 4097), (2, 12000), (256, 16384), (64, 16385), (2048, 16384), (2049, 16384), (4096, 700)])
@pytest.mark.parametrize("big", [0, 1, 3])
def test_sorting(ops, experts, pairs, big):
    ids = torch.randint(-1, experts + 1, (pairs,), generator=torch.Generator().manual_seed(pairs), dtype=torch.int32)
    by_expert, offsets, tiles, most = ops._pair_index(pairs, experts, big)
    by_expert.fill_(-7)
    on_device = ids.cuda()
    ops._call(
        "mlr_moe_align", ops._ptr(on_device), pairs, experts, big, most, ops._ptr(by_expert), ops._ptr(offsets), ops._ptr(tiles), ops._stream()
    )
    by_expert, offsets, tiles = by_expert.tolist(), offsets.tolist(), tiles.view(-1, 2).tolist()
    counts = torch.bincount(ids[(ids >= 0) & (ids < experts)].long(), minlength=experts)
    assert offsets == [0] + counts.cumsum(0).tolist()
    rows = ops.lib.mlr_moe_tile_rows(big)
    used = [[e, offsets[e] + i] for e in range(experts) for i in range(0, offsets[e + 1] - offsets[e], rows)]
    assert tiles == used + [[-1, len(used)]] * (most - len(used))
    mine = by_expert[: offsets[-1]]
    assert sorted(mine) == ((ids >= 0) & (ids < experts)).nonzero().flatten().tolist()
    assert all(ids[p] == e for e in range(experts) for p in mine[offsets[e] : offsets[e + 1]])
    assert by_expert[offsets[-1] :] == [-7] * (pairs - offsets[-1])


def test_routing_of_infinities_and_nan(ops):
    inf, nan = float("inf"), float("nan")
    z = torch.tensor([[nan, 1.0, 0.5, 2.0], [-inf, -inf, -inf, -inf], [nan] * 4, [inf, 1.0, nan, -inf]])
    ids, w = ops.route_experts(z.cuda(), None, top=2, groups=1, keep_groups=1, scale=1.0)
    # NaN is never chosen while there is a number; with none left the id stays in range
    assert ids.tolist() == [[3, 1], [0, 1], [0, 0], [0, 1]]
    assert torch.equal(w[1].cpu(), torch.zeros(2)) and w[3, 0].item() == 1.0


# rows an expert around the tiles of 16, 64, 128 and 256, one expert without rows; features around 64, 128 and 256; slices of 64 and 128 k
# and tails, one to seventeen slices of 64
@pytest.mark.parametrize("rows", [(1, 0, 15), (16, 17, 0), (63, 0, 65), (64, 129, 1), (127, 128, 0), (257, 3, 130), (191, 193, 256)])
@pytest.mark.parametrize("hidden,inner", [(8, 8), (72, 136), (520, 200), (1032, 264)])
@pytest.mark.parametrize("tiles", [0, 1, 2, 3])
def test_grouped_products(rows, hidden, inner, tiles):
    from mini_llm_runtime_amd.kernels.ops import HipOps
    from mini_llm_runtime_amd.kernels.tuning import KernelTuning

    never = 1 << 20
    tuning = KernelTuning(moe_tiled_rows=1 if tiles else never, moe_wide_tiled_rows=1 if tiles > 1 else never,
                          moe_square_groups=1 if tiles > 2 else never)
    ops = HipOps(torch.bfloat16, "cuda", tuning=tuning)
    experts, tokens = len(rows), sum(rows)
    h = _rand((tokens, hidden), torch.bfloat16, 81)
    up = _rand((experts * inner, hidden), torch.bfloat16, 82, hidden**-0.5)
    down = _rand((experts * hidden, inner), torch.bfloat16, 83, inner**-0.5)
    chosen = torch.repeat_interleave(torch.arange(experts), torch.tensor(rows))[torch.randperm(tokens, generator=torch.Generator().manual_seed(84))]
    ids = chosen.to(torch.int32)[:, None].contiguous()
    weights = torch.rand((tokens, 1), generator=torch.Generator().manual_seed(85)) + 0.5
    args = (h.cuda(), up.cuda(), down.cuda(), ids.cuda(), weights.cuda())
    got = ops.expert_products(*args, experts=experts, activation="relu2")[0].cpu().double()
    want, slack = torch.zeros(tokens, hidden, dtype=torch.double), torch.zeros(tokens, hidden, dtype=torch.double)
    for e in range(experts):
        of = (chosen == e).nonzero()[:, 0]
        u, d = up.double()[e * inner : (e + 1) * inner], down.double()[e * hidden : (e + 1) * hidden]
        x = h.double()[of]
        a = (x @ u.t()).clamp(min=0) ** 2
        # the hidden sums and their squares in float32, one rounding to bfloat16, the sums over inner in float32
        da = 2 * (x @ u.t()).abs() * hidden * 2.0**-24 * (x.abs() @ u.abs().t()) + 2.0**-8 * a + 1e-7
        pw = weights.double()[of]
        want[of] = pw * (a @ d.t())
        slack[of] = pw * (da @ d.abs().t() + (inner + 2) * 2.0**-24 * ((a + da) @ d.abs().t())) + 1e-7
    assert ((got - want).abs() <= slack).all()
    same = ops.expert_products(*args, experts=experts, activation="relu2")[0].cpu().double()
    assert torch.equal(got, same)


# matrices of a megabyte and more: whole lines through LDS; fewer slices of k than buffers and more, tails of k, features that end inside a tile
@pytest.mark.parametrize("rows", [(1, 0, 15), (16, 17, 0), (33, 1, 20)])
@pytest.mark.parametrize("hidden,inner", [(72, 8008), (8008, 72), (1160, 1032), (264, 2040)])
def test_products_that_stream_from_memory(rows, hidden, inner):
    test_grouped_products(rows, hidden, inner, 0)


@pytest.mark.parametrize("experts", [6, 8, 12, 16])  # 3, 4, 6 and 8 pairs of tiles: their features on eight, two, four dies and on one
@pytest.mark.parametrize("tiles", [1, 2, 3])
def test_few_tiles_on_all_dies(experts, tiles):
    test_grouped_products((20,) * experts, 1160, 1032, tiles)  # 10 and 9 runs of 128 features, 5 of 256: not the same number for every die


# experts of more rows than others make a tile or two more than whole rounds of dies hold: their features go to all dies
@pytest.mark.parametrize("more", [1, 2])
@pytest.mark.parametrize("tiles", [1, 2, 3])
def test_more_tiles_than_equal_shares_make(more, tiles):
    full = (0, 64, 128, 256)[tiles]
    test_grouped_products((full + 9,) * more + (full // 2,) * (16 - more), 1160, 264, tiles)


@pytest.mark.parametrize("inner", [4, 12, 72])  # 8, 24 and 144 woven rows: results of 8, 24 and 144 bytes (the second is stored directly)
@pytest.mark.parametrize("tiles", [1, 2, 3])
def test_gated_products_of_woven_rows(inner, tiles):
    """The gating in the epilogue is the plain product's, whatever the tile."""
    from mini_llm_runtime_amd.kernels.ops import HipOps
    from mini_llm_runtime_amd.kernels.tuning import KernelTuning

    never = 1 << 20
    tuning = KernelTuning(moe_tiled_rows=1, moe_wide_tiled_rows=1 if tiles > 1 else never, moe_square_groups=1 if tiles > 2 else never)
    experts, tokens, hidden = 3, 400, 136
    h = _rand((tokens, hidden), torch.bfloat16, 86).cuda()
    up = _rand((experts * 2 * inner, hidden), torch.bfloat16, 87, 0.2).cuda()
    down = _rand((experts * hidden, inner), torch.bfloat16, 88, 0.2).cuda()
    ids = torch.randint(0, experts, (tokens, 2), generator=torch.Generator().manual_seed(89)).to(torch.int32).cuda()
    weights = torch.ones((tokens, 2), device="cuda")
    kw = dict(experts=experts, activation="clamped_glu", glu=(7.0, 1.7), woven=True)
    got = HipOps(torch.bfloat16, "cuda", tuning=tuning).expert_products(h, up, down, ids, weights, **kw).double()
    want = HipOps(torch.bfloat16, "cuda").expert_products(h, up, down, ids, weights, kernel="fma", **kw).double()
    # an activation may round to the neighbouring bfloat16: 2^-8 of it (and another 2^-8 where the two gatings differ), times |down|
    act = torch.full((1,), 2.0**-7, dtype=torch.double, device="cuda")
    bound = act * 8.0 * 7.0 * down.double().abs().sum(-1).max()
    assert ((got - want).abs() <= bound).all() and ((got - want).norm() <= 2.0**-7 * want.norm())


# streaming from memory, streaming by whole lines (a matrix of a megabyte), tiles of 64, 128 and 256 rows
@pytest.mark.parametrize("kind,wide", [("16 rows", 16), ("16 rows", 256), ("64", 16), ("128", 16), ("256", 16)])
def test_inputs_beyond_two_gigabytes(kind, wide):
    """Input rows lie at 32-bit offsets of up to 4 GB: those at and behind 2 GB, where the mark for weights out of range lies, are rows like
    any other."""
    from mini_llm_runtime_amd.kernels.ops import HipOps
    from mini_llm_runtime_amd.kernels.tuning import KernelTuning

    far = 1 << 30
    ops = HipOps(torch.bfloat16, "cuda", tuning=KernelTuning(
        moe_tiled_rows=far if kind == "16 rows" else 1, moe_wide_tiled_rows=1 if kind in ("128", "256") else far,
        moe_square_groups=1 if kind == "256" else far))
    hidden, first = 2048, (1 << 31) // (2048 * 2)
    tokens = first + 40
    g = torch.Generator(device="cuda")
    g.manual_seed(85)
    h = torch.empty((tokens, hidden), dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    up, down = _rand((2 * wide, hidden), torch.bfloat16, 86, 0.05).cuda(), _rand((2 * hidden, wide), torch.bfloat16, 87, 0.2).cuda()
    ids = (torch.arange(tokens, dtype=torch.int32, device="cuda") % 2)[:, None].contiguous()
    weights = torch.ones((tokens, 1), device="cuda")
    out = ops.expert_products(h, up, down, ids, weights, experts=2, activation="relu2")[0]
    for e in (0, 1):
        rows = torch.arange(first - 2 + e, tokens, 2, device="cuda")
        z = h[rows].double() @ up[e * wide : (e + 1) * wide].double().t()
        act = z.clamp(min=0) ** 2
        want = act @ down[e * hidden : (e + 1) * hidden].double().t()
        # the activations are rounded to bfloat16 (2^-9 of themselves), everything else is float32
        bound = 2.0**-8 * act.abs() @ down[e * hidden : (e + 1) * hidden].double().abs().t() + 1e-3
        assert ((out[rows].double() - want).abs() <= bound).all()
