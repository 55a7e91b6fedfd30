"""What the attention kernels want to know about a batch before they are launched: the plan
a mixer that uses them hands to the step function, which uploads its arrays with the step's
other metadata and makes its sizes part of a recorded step's identity.
"""

from __future__ import annotations

import numpy as np

from ..parts.context import MixerPlan, PlanInput

QUERY_TILE = 64  # queries of one request that the prompt kernel takes together
WIDE_QUERY_TILE = 128  # and in its variant for long prompts (two blocks of queries per wavefront)
LONG_PREFIX_KEYS = 2048  # mean number of keys before a tile from which a step counts as behind long prefixes (twice: very long)
LONG_PROMPT_TILES = 12  # from which a prompt counts as long (see attention_f32.hip, groups_for)
GROUPED_TILES = 448  # wide tiles x heads of long prompts up to which they come in two groups of keys (see in_key_groups)
PAGED_ATTENTION = "paged_attention"  # the plan's key: every mixer on these kernels shares one plan per step


def query_tiles(q_lens, q_starts=None, tile: int = QUERY_TILE) -> np.ndarray:
    """[num_tiles, 2] int32 (entry, first query) covering every entry with more than one new
    token in tiles of `tile` queries, the tiles with the most keys before them first, those that see the most keys first
    among equals (a step of many short prompts has many first tiles, some of a few tokens): a kernel
    that hands them to the compute units in that order can start the heavy ones early and pair
    them with light ones.  Without the second order / with it, 32 heads of 128, 8 prompts of 43 to 329 tokens 22.0 / 18.7 us; over 280
    steps of 1 to 32 prompts at heads of 64 and 128, in both sizes of tiles, 0.996 of the time."""
    tiles = [(r, q0) for r, n in enumerate(q_lens) if n > 1 for q0 in range(0, int(n), tile)]
    if q_starts is None:
        q_starts = [0] * len(q_lens)
    tiles.sort(key=lambda t: (-(int(q_starts[t[0]]) + t[1]), -min(int(q_lens[t[0]]) - t[1], tile)))
    return np.asarray(tiles, dtype=np.int32).reshape(-1, 2)


def _coarse(n: int) -> int:
    """n rounded up to four binary digits: sizes of a plan are part of a recording's identity, and few recordings are kept."""
    unit = 1 << max(0, n.bit_length() - 4)
    return -(-n // unit) * unit


def attention_plan(shape: PlanInput) -> MixerPlan:
    """Tiles of 64 and of 128 queries over the entries with several new tokens (for the prompt
    kernel and its wide variant; the launch picks one by how many there are), how many of 64 the longest
    portion has (up to where it counts as long), for long portions that are not behind long prefixes the most keys that a
    wide tile of the step sees and the mean over its wide tiles, and
    how many entries have a single token and how long their contexts may be (for the split-KV
    decode kernel).  `shape.max_context` bounds the contexts; a recording is made with the
    capacity of its block tables there, so that it holds for every later step of its sizes."""
    single = shape.q_lens == 1
    decodes = int(single.sum())
    tiles = query_tiles(shape.q_lens, shape.q_starts)
    wide = query_tiles(shape.q_lens, shape.q_starts, WIDE_QUERY_TILE)
    # portions behind long cached prefixes: every tile has thousands of keys before it, so fewer
    # tiles keep the compute units busy for long and the wide tiles' lower cost per key wins
    # (level 1); behind twice as many (level 2) few tiles have their keys cut into runs
    keys_before = [int(shape.q_starts[e]) + int(q0) for e, q0 in wide]
    mean_before = sum(keys_before) / len(keys_before) if keys_before else 0
    long_prefix = int(mean_before >= LONG_PREFIX_KEYS) + int(mean_before >= 2 * LONG_PREFIX_KEYS)
    most_new = max((int(n) for n in shape.q_lens if n > 1), default=0)
    most_keys = mean_keys = 0
    if -(-most_new // QUERY_TILE) >= LONG_PROMPT_TILES and not long_prefix:
        keys = [int(shape.q_starts[e]) + min(int(q0) + WIDE_QUERY_TILE, int(shape.q_lens[e])) for e, q0 in wide]
        most_keys, mean_keys = _coarse(max(keys)), _coarse(sum(keys) // len(keys))
    return MixerPlan(
        key=PAGED_ATTENTION,
        arrays={"query_tiles": tiles, "wide_query_tiles": wide},
        sizes={
            "num_query_tiles": len(tiles),
            "num_wide_query_tiles": len(wide),
            "long_prefix": long_prefix,
            "longest_prompt_tiles": min(-(-most_new // QUERY_TILE), LONG_PROMPT_TILES),
            "most_prompt_keys": most_keys,
            "mean_prompt_keys": mean_keys,
            "num_decode_entries": decodes,
            "max_decode_context": int(shape.max_context) if decodes else 0,
        },
    )


def _prompt_keys(plan, num_tiles: int) -> tuple[int, int]:
    """The most keys that a wide tile sees and the mean; of a plan that does not say, as of one prompt."""
    most = int(getattr(plan, "most_prompt_keys", 0)) or QUERY_TILE * num_tiles
    return most, int(getattr(plan, "mean_prompt_keys", 0)) or (most + WIDE_QUERY_TILE) // 2


def long_chains(plan, num_tiles: int, reach: int) -> bool:
    """Whether a step's prompts make long chains of keys, the early tiles' shorter than the late ones': long prompts (the longest counts, however
    many there are), and a mask that reaches most of the longest (0: all of it)."""
    if int(getattr(plan, "longest_prompt_tiles", 0)) < LONG_PROMPT_TILES:
        return False
    return not reach or 4 * reach >= 3 * _prompt_keys(plan, num_tiles)[0]


def uneven_chains(plan, num_tiles: int) -> bool:
    """Whether the tiles' chains of keys run from short to long, as a whole prompt's do, instead of being long all alike behind cached tokens."""
    most, mean = _prompt_keys(plan, num_tiles)
    return 5 * mean <= 3 * most + 5 * QUERY_TILE


def in_key_groups(plan, num_tiles: int, groups: int, behind: int, window: int, chunk: int) -> bool:
    """Whether wide tiles of heads of 128 come with their keys in two groups (eight wavefronts, a workgroup to a compute unit) or in one (four,
    two workgroups); groups: wide tiles x heads.  In microseconds, one / two groups:
    Up to 256, one round: the chain is halved.  28 heads, 1,024 behind 4,096 112 / 90, 16 heads, 4 of 512 19.0 / 17.1, 8 of 256 13.8 / 13.4; not up
    to three tiles of keys, which end before the groups have met: 8 of 192 10.5 / 10.9, 16 of 128 11.4 / 11.7 (behind 300 cached tokens 20.9 / 22.3), 2,048
    in a window of 64 13.5 / 13.8 (of 80 15.5 / 14.6), in chunks of 128 11.6 / 11.9 (of 160 14.4 / 13.6).
    Beyond, where the second round is short: a unit takes some groups / 256 chains of the mean length one after the other, and at least the 256th
    and the 257th longest; in one group the longest decides.  1.4 most - 487 keys is where both took the same over 175 steps of whole prompts and
    behind some cached tokens: 28 heads, 2,048 53.9 / 49.4, twice 1,024 32.6 / 34.0, 1,024, 512 and 256 together 31.7 / 28.0, twice 896 29.2 / 30.2,
    twice 768 26.3 / 26.2; 32 heads, 1,596 42.0 / 38.1; 16 heads, 3,000 70 / 56; 64 heads, 760 behind 300 34.9 / 38.3; 40 heads, 1,000 behind 900 51.4 /
    56.6; 28 heads, 1,300 behind 500 48.6 / 44.6, 1,500 behind 1,200 68.1 / 70.6.  From 449 to 512 it would hold as well (28 heads, 2,304 61.2 / 57.2,
    twice 1,152 37.0 / 38.1), beyond there is a third round (28 heads, 2,432 65.9 / 67.3).  Behind long prefixes a second round is as long as the
    first: 28 heads, 1,500 behind 4,096 145 / 155."""
    if groups <= 256:
        tiles = int(getattr(plan, "longest_prompt_tiles", 0))  # 0: not known
        if behind:
            return True
        if 0 < (window or chunk) < 8 * QUERY_TILE:  # what a tile sees, cached tokens before it or not
            return window + WIDE_QUERY_TILE - 1 > 3 * QUERY_TILE if window else chunk > 2 * QUERY_TILE
        return not 0 < tiles <= 3
    most, mean = _prompt_keys(plan, num_tiles)
    if behind or groups > GROUPED_TILES or not long_chains(plan, num_tiles, window or chunk):
        return False
    return max(mean * groups / 256, 2 * most - 1024 * (most - mean) / groups) < 1.4 * most - 487
