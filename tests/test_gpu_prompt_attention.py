"""The 32 x 32 prompt attention (head sizes 64 and 128) at the edges of its tiles, against the plain 32-bit kernel."""

from __future__ import annotations

import pytest
import torch

from test_gpu_kernels import _attend, _paged_case, _rand, _tol

pytestmark = pytest.mark.gpu


# wide: four wavefronts; groups: the same tiles by eight in two groups of keys at heads of 128, whichever the launch would take (plans.in_key_groups)
@pytest.fixture(scope="module", params=["narrow", "wide", "groups"])
def ops(request):
    from mini_llm_runtime_amd.kernels.ops import HipOps
    from mini_llm_runtime_amd.kernels.tuning import KernelTuning

    if request.param != "narrow":
        form = 1 if request.param == "wide" else 2

        class OneForm(HipOps):
            def _call(self, name, *args, lib=None):
                if name == "mlr_attention_prefill" and args[8]:
                    args = (*args[:8], form, *args[9:])
                return super()._call(name, *args, lib=lib)

        return OneForm(torch.bfloat16, "cuda", tuning=KernelTuning(wide_attention_groups=1))
    return HipOps(torch.bfloat16, "cuda", tuning=KernelTuning(wide_attention_groups=1 << 30))


# queries around 32 (a wavefront), 64 and 128 (a workgroup); last keys at every kind of place among 8, 16 and 64; portions behind
# cached tokens; what no key was written to holds NaN
ENTRIES = [(2, 2), (31, 31), (33, 33), (64, 64), (65, 65), (127, 127), (129, 129), (200, 70), (331, 5), (192, 130), (77, 1)]


@pytest.mark.parametrize("heads,kv_heads,head_dim,block", [(14, 2, 64, 16), (4, 1, 128, 16), (3, 3, 64, 64), (2, 1, 128, 32)])
@pytest.mark.parametrize(
    "mask", [dict(window=None), dict(window=50), dict(window=None, chunk=48), dict(window=None, softcap=3.0)], ids=["causal", "window", "chunk", "cap"]
)
@pytest.mark.parametrize("sink", [False, True])
def test_edges(ops, heads, kv_heads, head_dim, block, mask, sink):
    q, kp, vp, table, ctx, *_ = _paged_case(ENTRIES, heads, kv_heads, head_dim, block, torch.bfloat16, 51, spike=True)
    args = (q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx)
    kw = dict(num_heads=heads, num_kv_heads=kv_heads, head_dim=head_dim, block_size=block, scale=head_dim**-0.5, **mask)
    if sink:
        kw["sinks"] = _rand((heads,), torch.float32, 52, 2.0).cuda()
    got, plain = _attend(ops, *args, **kw).cpu(), _attend(ops, *args, kernel="fma", **kw).cpu()
    assert torch.isfinite(got).all()
    torch.testing.assert_close(got.double(), plain.double(), **_tol(torch.bfloat16))


@pytest.mark.parametrize("head_dim", [64, 128])
def test_scores_that_keep_rising(ops, head_dim):
    """Every tile of keys scores higher than all before it, by a little and by much."""
    for step in (0.5, 4.0, 40.0):
        n = 300
        q, kp, vp, table, ctx, *_ = _paged_case([(n, n)], 2, 1, head_dim, 16, torch.bfloat16, 53)
        q[:, : 2 * head_dim] = 1.0
        for p in range(n):
            kp[table[0, p // 16], :, p % 16] = step * (p // 64) / head_dim + 0.01 * (p % 7)
        kw = dict(num_heads=2, num_kv_heads=1, head_dim=head_dim, block_size=16, scale=1.0, window=None)
        args = (q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx)
        got, plain = _attend(ops, *args, **kw).cpu(), _attend(ops, *args, kernel="fma", **kw).cpu()
        torch.testing.assert_close(got.double(), plain.double(), **_tol(torch.bfloat16))


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("entries", [[(6300, 200)], [(6300, 64)] * 5, [(9000, 16), (5000, 70)]])
@pytest.mark.parametrize("mask", [dict(window=None), dict(window=300), dict(window=1100), dict(window=None, chunk=700), dict(window=None, chunk=2000)])
def test_portions_behind_long_prefixes(ops, head_dim, entries, mask):
    """Keys in runs or whole, narrow tiles or wide ones, as what the mask lets a tile see and the tiles' number have it."""
    q, kp, vp, table, ctx, *_ = _paged_case(entries, 8, 2, head_dim, 16, torch.bfloat16, 57, spike=True)
    assert ctx.long_prefix == 2
    args = (q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx)
    kw = dict(num_heads=8, num_kv_heads=2, head_dim=head_dim, block_size=16, scale=head_dim**-0.5, **mask)
    got, plain = _attend(ops, *args, **kw).cpu(), _attend(ops, *args, kernel="fma", **kw).cpu()
    torch.testing.assert_close(got.double(), plain.double(), **_tol(torch.bfloat16))


@pytest.mark.parametrize("head_dim", [64, 128])
def test_a_key_that_outweighs_the_others(ops, head_dim):
    """A late key outweighs the first one by 2^7 to 2^8 and all others by 2^30, and both have the same values.  The largest weight is 1,
    which bfloat16 holds exactly, the first key's is at most 2^-7 and off by 2^-9 of that: the result is off by 2^-16, which rounds to the
    values themselves."""
    n, late = 192, 150
    q, kp, vp, table, ctx, *_ = _paged_case([(n, n)], 2, 1, head_dim, 16, torch.bfloat16, 55)
    values = _rand((head_dim,), torch.bfloat16, 56)
    kp[table[0].long()] = -40.0 / head_dim
    for p in (0, late):
        kp[table[0, p // 16], :, p % 16] = 0.0 if p == 0 else 8.0 / head_dim
        vp[table[0, p // 16], :, :, p % 16] = values
    # scores in powers of two (scale ln 2): 8 times the query's factor, between 7 and 8
    q[:, : 2 * head_dim] = (1.0 - torch.arange(n) % 32 / 256.0).bfloat16()[:, None]
    kw = dict(num_heads=2, num_kv_heads=1, head_dim=head_dim, block_size=16, scale=0.6931471805599453, window=None)
    got = _attend(ops, q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx, **kw).cpu()
    assert torch.equal(got[late:].view(n - late, 2, head_dim), values.expand(n - late, 2, head_dim))


# long prompts and portions whose tiles leave their sums for the merge that takes the pooled entries' share in: tiles without any, with few, with
# a part of a run past a page; one more query than a tile has
@pytest.mark.parametrize("heads,kv_heads,head_dim,block", [(4, 1, 128, 16), (6, 2, 64, 16), (2, 2, 128, 32)])
@pytest.mark.parametrize("window,pool", [(300, 4), (65, 7)])
@pytest.mark.parametrize("sink", [False, True])
def test_pooled_entries_beside_the_tiles(ops, heads, kv_heads, head_dim, block, window, pool, sink):
    entries = [(1300, 1300), (900, 129), (331, 5), (64, 64), (700, 1)]
    q, kp, vp, table, ctx, *_ = _paged_case(entries, heads, kv_heads, head_dim, block, torch.bfloat16, 62)
    pooled_kp, pooled_vp, pooled_table = _paged_case([(-(-c // pool), 1) for c, _ in entries], heads, kv_heads, head_dim, block, torch.bfloat16, 63)[1:4]
    kw = dict(num_heads=heads, num_kv_heads=kv_heads, head_dim=head_dim, block_size=block, scale=head_dim**-0.5, window=window)
    kw["pooled"] = (pooled_kp.cuda(), pooled_vp.cuda(), pooled_table.cuda(), pool)
    if sink:
        kw["sinks"] = _rand((heads,), torch.float32, 64, 2.0).cuda()
    args = (q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx)
    got, plain = _attend(ops, *args, **kw).cpu(), _attend(ops, *args, kernel="fma", **kw).cpu()
    assert torch.isfinite(plain).all()
    torch.testing.assert_close(got.double(), plain.double(), **_tol(torch.bfloat16))


# workgroups (entries x heads) around one and two to every compute unit, and many more; entries of unequal contexts
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("entries", [63, 64, 65, 127, 128, 129, 200])
def test_every_workgroup_has_its_work(ops, head_dim, entries):
    lens = [(2 + 3 * i % 50, 2) for i in range(entries)]
    q, kp, vp, table, ctx, *_ = _paged_case(lens, 4, 2, head_dim, 16, torch.bfloat16, 59)
    kw = dict(num_heads=4, num_kv_heads=2, head_dim=head_dim, block_size=16, scale=head_dim**-0.5, window=None)
    args = (q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx)
    got, plain = _attend(ops, *args, **kw).cpu(), _attend(ops, *args, kernel="fma", **kw).cpu()
    torch.testing.assert_close(got.double(), plain.double(), **_tol(torch.bfloat16))


# two rounds of narrow tiles or one of wide ones: long prompts up to 512 narrow tiles x heads, short ones, one tile more, masks that reach
# three quarters of the prompts and less, cached tokens before them; 2: wide tiles in two groups of keys, up to 256 of them or 448 of long prompts
@pytest.mark.parametrize(
    "heads,entries,mask,wide",
    [
        (8, [(4096, 4096)], {}, 0), (16, [(2100, 2100)], {}, 2), (16, [(1024, 1024)] * 2, {}, 0), (16, [(704, 704)] * 2 + [(640, 640)], {}, 1),
        (8, [(4096, 4096)], dict(window=3072), 0), (8, [(4096, 4096)], dict(chunk=3071), 2), (16, [(4100, 2048)], {}, 2),
        (28, [(2048, 2048)], {}, 2), (28, [(2049, 2049)], {}, 1), (28, [(2048, 2048)], dict(window=1000), 1), (16, [(4200, 2049)], {}, 1),
    ],
)
def test_two_rounds_of_narrow_tiles(heads, entries, mask, wide):
    from mini_llm_runtime_amd.kernels.ops import HipOps

    launches = []

    class Spying(HipOps):
        def _call(self, name, *args, lib=None):
            if name == "mlr_attention_prefill":
                launches.append(int(args[8]))
            return super()._call(name, *args, lib=lib)

    ops = Spying(torch.bfloat16, "cuda")
    q, kp, vp, table, ctx, *_ = _paged_case(entries, heads, 1, 128, 16, torch.bfloat16, 60)
    ctx.longest_prompt_tiles = min(12, max(-(-n // 64) for _, n in entries))
    kw = dict(num_heads=heads, num_kv_heads=1, head_dim=128, block_size=16, scale=128**-0.5, **{"window": None, **mask})
    args = (q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx)
    got, plain = _attend(ops, *args, **kw).cpu(), _attend(ops, *args, kernel="fma", **kw).cpu()
    assert launches == [wide]
    torch.testing.assert_close(got.double(), plain.double(), **_tol(torch.bfloat16))


# prompts in one step under a mask that reaches all of each, and long portions whose tiles all have cached tokens before them
@pytest.mark.parametrize(
    "heads,entries,mask,wide",
    [(16, [(1792, 1792)] * 2, dict(window=1792), 2), (16, [(1792, 1792)] * 2, dict(window=1100), 1), (16, [(1024, 1024)] * 2, dict(chunk=1024), 0),
     (32, [(2500, 1000)], {}, 2), (32, [(1100, 1000)], {}, 0)],
)
def test_forms_by_the_longest_prompt(heads, entries, mask, wide):
    _check_form(heads, entries, mask, wide)


# wide tiles in one group of keys or two: one round and chains of three key tiles or more, short ones behind masks; two rounds of long prompts whose
# chains are long enough for their number, alike or not, of portions with few and with many cached tokens
@pytest.mark.parametrize(
    "heads,entries,mask,wide",
    [
        (16, [(192, 192)] * 8, {}, 1), (16, [(256, 256)] * 8, {}, 2), (16, [(128, 128)] * 16, dict(window=4096), 1), (16, [(256, 256)] * 8, dict(chunk=512), 2), (8, [(600, 128)] * 32, {}, 1), (16, [(2048, 2048)], dict(window=65), 1),
        (16, [(2048, 2048)], dict(window=66), 2), (16, [(2048, 2048)], dict(chunk=128), 1), (16, [(2048, 2048)], dict(chunk=160), 2),
        (28, [(1024, 1024)] * 2, {}, 1), (28, [(1024, 1024), (512, 512), (256, 256)], {}, 2), (28, [(896, 896)] * 2, {}, 1), (28, [(1280, 1280)], {}, 2),
        (40, [(1900, 1000)], {}, 1), (28, [(1800, 1300)], {}, 2), (28, [(2048, 2048)], {}, 2), (28, [(2049, 2049)], {}, 1),
    ],
)
def test_one_group_of_keys_or_two(heads, entries, mask, wide):
    _check_form(heads, entries, mask, wide)


def _check_form(heads, entries, mask, wide):
    """The form that the launch takes for a step with this plan (as in the test above), and its result."""
    import numpy as np

    from mini_llm_runtime_amd.kernels.ops import HipOps
    from mini_llm_runtime_amd.kernels.plans import attention_plan
    from mini_llm_runtime_amd.parts.context import PlanInput

    launches = []

    class Spying(HipOps):
        def _call(self, name, *args, lib=None):
            if name == "mlr_attention_prefill":
                launches.append(int(args[8]))
            return super()._call(name, *args, lib=lib)

    ops = Spying(torch.bfloat16, "cuda")
    q, kp, vp, table, ctx, *_ = _paged_case(entries, heads, 1, 128, 16, torch.bfloat16, 61)
    lens, starts = [np.array(n, dtype=np.int32) for n in ([n for _, n in entries], [c - n for c, n in entries])]
    for name, value in attention_plan(PlanInput(lens, starts, max(c for c, _ in entries))).sizes.items():
        setattr(ctx, name, value)
    kw = dict(num_heads=heads, num_kv_heads=1, head_dim=128, block_size=16, scale=128**-0.5, **{"window": None, **mask})
    args = (q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx)
    got, plain = _attend(ops, *args, **kw).cpu(), _attend(ops, *args, kernel="fma", **kw).cpu()
    assert launches == [wide]
    torch.testing.assert_close(got.double(), plain.double(), **_tol(torch.bfloat16))


def test_a_page_that_is_not_there(ops):
    q, kp, vp, table, ctx, *_ = _paged_case([(100, 100), (300, 300)], 2, 1, 64, 16, torch.bfloat16, 54)
    table = table.clone()
    table[1, 9] = -1  # positions 144..159 of the second request
    kw = dict(num_heads=2, num_kv_heads=1, head_dim=64, block_size=16, scale=0.125, window=None)
    got = _attend(ops, q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx, **kw).cpu()
    assert torch.isfinite(got[:228]).all() and torch.isnan(got[100 + 256 :]).all()


def give_back(entries, kp, vp, table, block, window=None, chunk=None):
    """The table and pages once every page wholly before the first visible key of a request's next token has been given back: its entry
    is -1, and somebody else has written what has no value there."""
    table, kp, vp = table.clone(), kp.clone(), vp.clone()
    gone = 0
    for r, (context, new) in enumerate(entries):
        p = context - new
        first = p // chunk * chunk if chunk else max(0, p - window + 1)
        for page in range(first // block):
            kp[table[r, page]] = vp[table[r, page]] = float("nan")
            table[r, page] = -1
            gone += 1
    assert gone
    return kp, vp, table


# first visible keys at the start of a tile of 64 keys, at its end and inside, of a page and of 16 keys of a larger page
@pytest.mark.parametrize("heads,kv_heads,head_dim,block", [(4, 2, 64, 16), (2, 1, 128, 16), (2, 2, 64, 64), (2, 1, 128, 32)])
@pytest.mark.parametrize("mask", [dict(window=1), dict(window=17), dict(window=50), dict(window=65), dict(window=None, chunk=48), dict(window=None, chunk=160)])
def test_pages_that_were_given_back(ops, heads, kv_heads, head_dim, block, mask):
    entries = [(200, 70), (331, 5), (192, 130), (385, 129), (448, 64), (403, 140)]
    q, kp, vp, table, ctx, *_ = _paged_case(entries, heads, kv_heads, head_dim, block, torch.bfloat16, 58)
    kw = dict(num_heads=heads, num_kv_heads=kv_heads, head_dim=head_dim, block_size=block, scale=head_dim**-0.5, **mask)
    whole = _attend(ops, q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), ctx, **kw).cpu()
    left = give_back(entries, kp, vp, table, block, **mask)
    got = _attend(ops, q.cuda(), *(t.cuda() for t in left), ctx, **kw).cpu()
    assert torch.isfinite(whole).all() and torch.equal(got, whole)
