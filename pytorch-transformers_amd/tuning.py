"""Choices between ways to the same result that are timed rather than ruled, and the table that keeps them.

Some choices have no rule that holds across shapes: how many ranges of K a pair launch is cut into, up to how many
rows the decode batch kernel beats the vendor library, in which pieces along M the library's product runs, whether
two matrices of one input run as one product, whether K is cut into a batch, and how a decode step's attention
launch is cut (for which there is a fitted model of the launch's time, below, that the timing may overrule).  Each
has a built-in default and an entry per shape in a ``TuningTable`` that overrides it.  A table is filled only while
timing is switched on: inside ``live_tuning()`` (``CausalLM.tune`` runs steps of given sizes in it), or in every
step with PTA_TUNE=1 in the environment.  With timing off (the default) a step allocates nothing for measurements
and times nothing, and its results depend on weights, tokens, schedule and table alone: two processes give the
same bits.  ``TuningTable.to_dict`` / ``load`` carry a table from one process to another.

``ops`` holds the kernel faces and asks here; this module calls the faces back when it times them.  The names of
this module are also reachable as attributes of ``ops``.
"""
from __future__ import annotations

import copy
import functools
import os
from typing import Optional

import torch

from . import ops


class TuningTable:
    """The choices that were timed rather than ruled, by shape.  A model owns one (``CausalLM.tuning``); callers of
    the kernel faces that bring none share ``DEFAULT``.  The table whose choices hold is the active one
    (``activate``): a model activates its own at the start of every step, so two models in one process neither see
    nor overwrite each other's choices.  The ranges of K of pair launches are also kept inside the kernel library,
    by shape; ``activate`` takes the old table's out of it and puts the new one's in."""

    FIELDS = ("pair_parts", "pair_stationary", "splitk_rows", "mm_plans", "mm_joined", "mm_ksplit", "mm_tiles", "decode_plans")

    def __init__(self, data: Optional[dict] = None):
        # (shape of w1, shape of w2) -> (ranges, ranges, row tiles per wave) in use, and another three where steps of 33 to 64
        # rows have theirs
        self.pair_parts: dict = {}
        # (shape of w1, shape of w2) -> per class of rows the (ranges, ranges) of the launch with stationary
        # activations, (0, 0) where the staged kernel stays
        self.pair_stationary: dict = {}
        self.splitk_rows: dict = {}  # ((N, K), ...) -> rows up to which the batch kernel beats the library's product
        self.mm_times: dict = {}  # (N, K) -> {rows: microseconds}; measurements, not part of the table as data
        self.mm_plans: dict = {}  # (N, K, M bucket) -> [rows, ...]
        self.mm_costs: dict = {}  # (N, K, M bucket) -> microseconds of that plan, as measured piece by piece
        # (N1, N2, K, M bucket), then (activation, bias) of each where there is any -> whether one product with both
        # matrices beats the two
        self.mm_joined: dict = {}
        self.mm_ksplit: dict = {}  # (N, K, M bucket) -> ranges of K (1: the plain product)
        # (N, K, M bucket, activation, bias, additions) -> whether the hand-written kernel beats the library's product
        self.mm_tiles: dict = {}
        self.decode_plans: dict = {}  # (batch, heads, KV heads, head size, longest, mean) as counted -> a timed cut
        if data:
            self.load(data)

    def to_dict(self) -> dict:
        """The table as plain data (JSON-able): loaded in another process, that process makes the same choices,
        hence the same bits."""
        key = lambda t: ",".join("x".join(str(int(v)) for v in (p if isinstance(p, tuple) else (p,))) for p in t)
        return {
            "pair_parts": {key(k): list(v) for k, v in self.pair_parts.items()},  # ranges, ranges, row tiles per wave (and again)
            "pair_stationary": {key(k): [list(c) for c in v] for k, v in self.pair_stationary.items()},  # per class of rows
            "splitk_rows": {key(k): int(v) for k, v in self.splitk_rows.items()},
            "mm_plans": {key(k): list(v) for k, v in self.mm_plans.items()},
            "mm_joined": {key(k): bool(v) for k, v in self.mm_joined.items()},
            "mm_ksplit": {key(k): int(v) for k, v in self.mm_ksplit.items()},
            "mm_tiles": {key(k): bool(v) for k, v in self.mm_tiles.items()},
            "decode_plans": {key(k): list(v) for k, v in self.decode_plans.items()},  # tiles, keys per workgroup, waves
        }

    def load(self, data: dict) -> None:
        """Take the choices of a table that ``to_dict`` made (entries for other shapes stay as they are).  The table
        becomes the active one, so that what it says about pair launches is checked by the kernel library now."""
        unknown = sorted(set(data) - set(self.FIELDS))
        if unknown:
            raise ValueError(f"a tuning table has the sections {list(self.FIELDS)}; this one also holds {unknown}")
        activate(self)
        _note_change()
        shapes = lambda k: tuple(tuple(int(v) for v in p.split("x")) for p in k.split(","))
        flat = lambda k: tuple(int(p) for p in k.split(","))
        for k, v in data.get("pair_parts", {}).items():
            s1, s2 = shapes(k)
            cut = tuple(int(n) for n in v) if len(v) != 2 else (int(v[0]), int(v[1]), 1)
            _fix_pair(s1, s2, cut)
            self.pair_parts[(s1, s2)] = cut
        for k, v in data.get("pair_stationary", {}).items():
            s1, s2 = shapes(k)
            cuts = tuple((int(c[0]), int(c[1])) for c in v)
            _fix_stationary(s1, s2, cuts)
            self.pair_stationary[(s1, s2)] = cuts
        for k, v in data.get("splitk_rows", {}).items():
            self.splitk_rows[shapes(k)] = int(v)
        for k, v in data.get("mm_plans", {}).items():
            self.mm_plans[flat(k)] = [int(r) for r in v]
        for k, v in data.get("mm_joined", {}).items():
            self.mm_joined[flat(k)] = bool(v)
        for k, v in data.get("mm_ksplit", {}).items():
            self.mm_ksplit[flat(k)] = int(v)
        for k, v in data.get("mm_tiles", {}).items():
            self.mm_tiles[flat(k)] = bool(v)
        for k, v in data.get("decode_plans", {}).items():
            self.decode_plans[flat(k)] = tuple(int(p) for p in v)

    def clear(self) -> None:
        """Back to the built-in defaults for every shape."""
        _note_change()
        if self is _active:
            _release(self)
        for d in (self.pair_stationary, self.pair_parts, self.splitk_rows, self.mm_plans, self.mm_costs, self.mm_times,
                  self.mm_joined, self.mm_ksplit, self.mm_tiles, self.decode_plans):
            d.clear()


_changes = 0  # times that a choice of some table was set or may have been timed


def changes() -> int:
    """A number that grows when choices change: what ran under another number may have run otherwise."""
    return _changes


def _note_change() -> None:
    global _changes
    _changes += 1


def _unfix_pair(s1, s2) -> None:
    ops.load_library().pta_gemm_splitk_pair_fix(int(s1[0]), int(s1[1]), int(s2[0]), int(s2[1]), 0, 0, 1)


def _fix_pair(s1, s2, cut) -> None:
    """Fix (ranges, ranges, row tiles per wave) for a pair of shapes in the kernel library, and the second three for steps of 33
    to 64 rows: also where they are the rule's for some rows, which has others for those."""
    lib, shapes = ops.load_library(), (int(s1[0]), int(s1[1]), int(s2[0]), int(s2[1]))
    refused = len(cut) not in (3, 6) or lib.pta_gemm_splitk_pair_fix(*shapes, *(int(n) for n in cut[:3]))
    if not refused and len(cut) == 6:
        refused = lib.pta_gemm_splitk_pair_fix_middle(*shapes, *(int(n) for n in cut[3:]))
    if refused:
        raise ops.KernelError(f"tuning table: ranges of K and row tiles {tuple(cut)} are not valid for the pair {tuple(s1)}, {tuple(s2)}")


def _fix_stationary(s1, s2, cuts) -> None:
    lib = ops.load_library()
    for cls, c in enumerate(cuts):
        if lib.pta_gemm_splitk_pair_fix_stationary(int(s1[0]), int(s1[1]), int(s2[0]), int(s2[1]), cls, int(c[0]), int(c[1])):
            raise ops.KernelError(f"tuning table: {list(c)} is not valid for the pair {tuple(s1)}, {tuple(s2)} with "
                                  "stationary activations")


def _release(table: "TuningTable") -> None:
    """Take what ``table`` fixed for pair launches out of the kernel library."""
    if not table.pair_parts and not table.pair_stationary:
        return
    lib = ops.load_library()
    for (s1, s2) in table.pair_parts:
        _unfix_pair(s1, s2)
    for (s1, s2) in table.pair_stationary:
        lib.pta_gemm_splitk_pair_fix_stationary(int(s1[0]), int(s1[1]), int(s2[0]), int(s2[1]), -1, 0, 0)


def _apply(table: "TuningTable") -> None:
    for (s1, s2), cut in table.pair_parts.items():
        _fix_pair(s1, s2, cut)
    for (s1, s2), cuts in table.pair_stationary.items():
        _fix_stationary(s1, s2, cuts)


DEFAULT = TuningTable()  # of whoever calls the kernel faces without a table of their own
_active = DEFAULT


def active() -> TuningTable:
    return _active


def activate(table: Optional[TuningTable]) -> TuningTable:
    """Make ``table`` (None: ``DEFAULT``) the one whose choices hold, and the one that timing fills."""
    global _active
    table = DEFAULT if table is None else table
    if table is not _active:
        _release(_active)
        _active = table
        _apply(table)
    return table


def tuning_table() -> dict:
    """The active table as plain data."""
    return _active.to_dict()


def clear_tuning() -> None:
    """The active table back to the built-in defaults for every shape."""
    _active.clear()


def load_tuning(table: dict) -> None:
    """Take a table's choices into the active one."""
    _active.load(table)


# ---- the cut of a decode step's attention launch --------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _decode_plan(n: int, n_heads: int, n_kv_heads: int, head_dim: int, bound: int, mean: int, most_tiles: int):
    """The cheapest cut of a decode launch of ``n`` sequences of up to ``bound`` keys, ``mean`` on average,
    by a model of its time.

    A wave holds ``t`` groups of sixteen heads of one KV head and walks ``size`` keys in blocks of 32.  In
    microseconds, fitted to launches with cold caches at three head shapes (71 heads on 1 KV head of 64; 32 on
    8 of 128; 128 on 8 of 64), 1 to 64 sequences of 1,100 to 8,192 keys, every cut (the model's choice is
    within a tenth of the best measured cut nearly everywhere, and mostly equal to it):

    - a wave takes 0.22 + 0.21 t + 0.15 (head_dim / 64 - 1) per block, and waves beyond what the chip
      holds at once (1,024 SIMDs, as many waves each as 512 registers allow) wait for a whole round;
    - the keys and values stream at 5.1 TB/s, and again at 7.2 TB/s for every further wave that shares
      a KV head;
    - the launch takes the 4.2-norm of those two times (the larger one, and more where they are close);
    - ranges cost 2.2 + 0.1 per range, and their partial sums (32-bit, written and read) move at 3.5 TB/s.

    The longest context of a step that is sized for ``bound`` lies in its last 1,024 and the mean in the 512
    below ``mean``, so the longest wave's time is taken at ``bound - 512`` keys and the traffic at
    ``mean - 256`` keys a sequence."""
    groups = (n_heads // n_kv_heads + 15) // 16
    dt = head_dim / 16.0
    keys = bound - 512
    mean_keys = min(keys, mean - 256)
    kv_mb = n * mean_keys * n_kv_heads * head_dim * 4 / 1e6
    best = None
    for t in range(1, most_tiles + 1):
        if ops.ATTN_FORCE_TILES and t != min(ops.ATTN_FORCE_TILES, most_tiles):
            continue
        sharing = (groups + t - 1) // t
        resident = 1024 * max(1, int(512 // ((38 + 11.5 * dt) + (26 + 8 * dt) * t)))
        block_us = 0.22 + 0.21 * t + 0.15 * (head_dim / 64.0 - 1.0)
        size = min(ops.ATTN_SPLIT_KEYS, ops.ATTN_FORCE_SPLIT) if ops.ATTN_FORCE_SPLIT else ops.ATTN_SPLIT_KEYS
        while True:
            whole = size >= bound
            if (bound + size - 1) // size <= 1024 and n * ((bound + size - 1) // size) <= 65535 and (not ops.ATTN_FORCE_SPLIT or size == ops.ATTN_FORCE_SPLIT or
                                                       (whole and size < ops.ATTN_FORCE_SPLIT)):
                ranges = (mean_keys + size - 1) // size
                waves = n * n_kv_heads * sharing * ranges
                wave_us = min(size, keys) / 32 * block_us * ((waves + resident - 1) // resident)
                stream_us = kv_mb / 5.1 + kv_mb * (sharing - 1) / 7.2
                part_us = 0.0 if whole else 2.2 + 0.1 * ranges + n * n_heads * ranges * head_dim * 8 / 1e6 / 3.5
                cost = (wave_us ** 4.2 + stream_us ** 4.2) ** (1 / 4.2) + part_us
                if best is None or cost < best[0]:
                    best = (cost, t, size)
            if whole:
                break
            size *= 2
    if best is None:
        raise ops.KernelError(f"no cut of a decode launch over {bound} keys with PTA_ATTN_SPLIT={ops.ATTN_FORCE_SPLIT}")
    return best[1], best[2]




# Decode launches over contexts up to here walk the whole context with one wave per sequence and group of sixteen heads, which
# leaves no ranges to merge; nothing is timed and no table is asked there.  Launch and merge, replayed over sixteen caches in
# turn, the ranges of ``decode_plan`` -> whole: 71 heads on 1 KV head of 64, 8 sequences of 64 / 130 / 300 / 500 keys 6.9 ->
# 3.5, 7.9 -> 4.9, 8.3 -> 7.1, 8.6 -> 9.2 us, 64 sequences 9.7 -> 4.8, 11.7 -> 6.5, 13.0 -> 8.4, 13.5 -> 11.5; 13 on 13 of 80, 5
# sequences 7.0 -> 4.1, 8.6 -> 6.2, 8.9 -> 7.9, 9.3 -> 10.2; 16 on 8 of 128, 2 sequences 6.6 -> 4.0, 7.4 -> 5.6, 8.6 -> 8.5,
# 8.7 -> 11.4; 128 on 8 of 64, 32 sequences 8.7 -> 4.3, 10.0 -> 5.7, 12.7 -> 8.9, 15.4 -> 13.2: the merge costs a launch,
# which few keys do not win back.  In whole steps, where keys come from memory, a lone wave on 300 keys is no longer the faster
# one (24 layers of 13 heads of 80 with ALiBi, 17 to 325 keys: 34.7 ms a request with ranges, 35.4 with whole contexts up to
# 320), at 60 keys it is by what the merge costs (32 layers of 71 heads, one sequence: 79.7 -> 77.1 ms).
SHORT_CONTEXT = 192


def context_bound(max_len: int) -> int:
    """The context that a captured decode step is sized for: ``SHORT_CONTEXT``, or the next multiple of 1,024."""
    return SHORT_CONTEXT if max_len <= SHORT_CONTEXT else (max_len + 1023) // 1024 * 1024


def short_cut(max_len: int):
    """The cut of a decode launch over so short a context (as ``decode_plan`` gives cuts), or None where it is longer."""
    if max_len > SHORT_CONTEXT or ops.ATTN_FORCE_SPLIT or ops.ATTN_FORCE_TILES:
        return None
    return (1, SHORT_CONTEXT, 1)


def decode_key(n_seqs: int, n_heads: int, n_kv_heads: int, head_dim: int, max_len: int, mean_len: int):
    n = 1
    while n < n_seqs:
        n *= 2
    bound = (max_len + 1023) // 1024 * 1024
    mean = min(bound, (mean_len + 511) // 512 * 512) if mean_len > 0 else bound
    return (n, int(n_heads), int(n_kv_heads), int(head_dim), bound, mean)


def late_waves(n_seqs: int, n_heads: int, n_kv_heads: int, head_dim: int, max_len: int, mean_len: int = 0) -> int:
    """0, or the waves (1 or 4) on the keys of sixteen heads with which a decode step's attention goes in the launch of the products behind it,
    where there is such a launch (``ops.gemm_splitk_pair_attn``) and its products leave the room (``late_pays``).  Whole contexts: a piece,
    sixteen heads of a KV head, occupies a workgroup, or a wave of one, for as long as its keys take behind the stream of weights, and every
    workgroup of attention is one less for that stream.  Microseconds a layer against launches apart, one wave / four:

                                        1 sequence       8               16              32              64
        71 heads on 1 of 64, 60 keys    -2.3 / -2.3   -1.3 / -0.1     -0.3 / +0.8     +0.6 / +2.3     -0.8 / +0.6
                            150 keys    -3.1 / -3.4   -2.6 / -0.8     -1.5 / +0.9     -1.3 / +0.9     +1.2 / +0.5
                            900 keys    +4.5 / -5.3    +11 / -3.8     +9.9 / +0.1     +7.7 / +0.9      +12 / +2.3
                          1,900 keys     +38 / -6.4    +48 / -5.5      +47 / +2.5      +45 / +4.6      +48 / +16
        128 on 8 of 64, 60 keys         -1.4 / -1.3   -1.2 / -0.3     +0.7 / +0.4     +1.5 / +0.7     -2.0 / +3.3
                       150 keys         -1.1 / -2.8   -0.4 / -0.8     +2.6 / -0.5     +2.2 / -0.5     +0.3 / +4.5
                       900 keys          +10 / -3.1    +12 / -1.2     +7.7 / -4.7      +13 / -0.9     +6.2 / +5.5
                     1,900 keys          +29 / +1.7    +27 / +2.7      +27 / +1.6      +15 / -9.5     +4.4 / +2.9

    So a wave alone up to ``SHORT_CONTEXT``, which is the cut of the launch apart there (``short_cut``), so that a result is the same whether it rides: with
    up to 320 pieces where the heads of a KV head fill several (whose waves share its keys), with up to 64 where a KV head is one: at 30 / 100 / 190 keys 128 on 8
    of 1 sequence -2.1 / -1.4 / -2.9 (four waves -1.7 / -3.1 / -3.4), of 8 -1.3 / -0.6 / -1.0 (-0.6 / -1.0 / -1.5), of 12 +0.0 / +1.8 / -0.1; 48 on 6 of 8 -1.1 / -2.3 / -3.6
    (-0.6 / -1.3 / -2.6).  Beyond that four waves, up to 2,048 keys where there are few pieces of several a KV head, up to 1,024 where a KV head is one piece.  (One
    answer for 33 to 64 sequences: 40 to 56 of 30 to 190 keys are -1.0 to -4.7, 64 from -0.8 to +3.0.)  A cut that was fixed (``set_decode_plan``) goes
    before the rule."""
    key = decode_key(n_seqs, n_heads, n_kv_heads, head_dim, max_len, mean_len)
    if ops.ATTN_FORCE_SPLIT or ops.ATTN_FORCE_TILES:
        return 0
    n, bound = key[0], key[4]
    groups = (n_heads // n_kv_heads + 15) // 16
    pieces = n * n_kv_heads * groups
    if max_len <= SHORT_CONTEXT:
        return 1 if pieces <= (320 if groups > 1 else 64) else 0
    cut = _active.decode_plans.get(key)
    if cut is not None:
        return 4 if cut[0] == 1 and cut[1] >= max_len and cut[2] == 4 else 0
    return 4 if (bound <= 2048 and pieces <= 40 if groups > 1 else bound <= 1024 and pieces <= 256) else 0


def late_pays(n_seqs: int, n_heads: int, n_kv_heads: int, head_dim: int, max_len: int, mean_len: int, rounds: int, slack: int) -> bool:
    """Whether the products of a pair's launch hide the attention that ``late_waves`` would have it carry: the second's workgroups wait for it, and the
    launch ends later where they have as much to do as the first's.  ``slack``: the blocks of a third of a microsecond that a compute unit has
    less of theirs; ``rounds``: the workgroups a unit has.  Microseconds a layer against launches apart, 1 / 8 / 32 sequences, by slack:

        150 keys   0: +0.1 / +1.1 / +2.1 (of 28 to 31)    11: -3.0 / -1.5 / -1.5 (of 40)    16: -3.4 / -2.9 / -2.0 (of 20)    22: -4.2 / -1.9 / -1.8 (of 42)
        500        0: +1.1 / +2.2 / +4.0                  11: -1.5 / +0.8 / +1.5            16: -2.1 / -1.2 / -0.6            22: -3.6 / -0.8 / -0.7
        900        0: +4.4 / +5.0 / +4.8                  16: +0.7 / +1.8 / +1.9            22: -1.3 / +0.9 / +2.5            32: -3.2 / -0.6 / -0.8
        1,900      0: +13 / +13 / +13                     22: +6.6 / +6.8 / +11             48: +1.4 / +1.3                   154: -6.4 / -5.5 / +4.6

    So 8 blocks for a short context, 16 for one of 512 keys on average and 20 beyond, 64 past 1,024 keys.  The 11 and 16 are of four waves on the keys of a KV head
    of one piece, which take one up to ``SHORT_CONTEXT`` and want 16 then: at 150 keys 11: +0.2 / +1.2, 16: -3.2 / +0.5 (of 20), 22: -1.2 / +0.0.  Few pieces
    beside two workgroups a unit find room without: 96 heads on 8, 480 workgroups, one sequence -2.0 at 30 keys to -5.0 at 900; 80 on 1, 8 sequences, +0.0 to +0.5."""
    n, _, _, _, bound, mean = decode_key(n_seqs, n_heads, n_kv_heads, head_dim, max_len, mean_len)
    groups = (n_heads // n_kv_heads + 15) // 16
    pieces = n * n_kv_heads * groups
    if rounds > 1 and pieces <= 40 and bound <= 1024:
        return True
    if max_len <= SHORT_CONTEXT:
        return slack >= (8 if groups > 1 else 16)
    return slack >= (64 if bound > 1024 else 16 if mean <= 512 else 20)


def decode_plan(n_seqs: int, n_heads: int, n_kv_heads: int, head_dim: int, max_len: int, mean_len: int = 0):
    """How a decode launch is cut: (column tiles per wave, keys per workgroup, waves per workgroup); a size that
    covers the context means one workgroup per sequence and head group, which writes the result itself.  The
    waves of a workgroup take its keys block by block in turn and merge in LDS; ``SHARED_KEYS`` in their place
    means a wave per tile of heads, all on the same keys (``_shared_keys_rule``).

    The batch counts by its next power of two, the longest context by its next multiple of 1,024 and the
    mean context (``mean_len``; 0: as the longest) by its next multiple of 512, so that a captured step,
    which is sized for a padded batch and such bounds, is cut exactly as the same step run directly.
    A cut that was fixed for these counts (``set_decode_plan``; ``CausalLM.tune`` times whole steps with the cuts
    of ``decode_plan_candidates``) goes before the rule, which has one wave per workgroup or shared keys."""
    key = decode_key(n_seqs, n_heads, n_kv_heads, head_dim, max_len, mean_len)
    kept = _active.decode_plans.get(key)
    if kept is not None:
        return kept
    n, _, _, _, bound, mean = key
    shared = _shared_keys_rule(n, n_heads, n_kv_heads, head_dim, bound, mean)
    if shared is not None:
        return shared
    groups = (n_heads // n_kv_heads + 15) // 16
    most = min(groups, int(ops.load_library().pta_attn_decode_max_tiles(head_dim)))
    return _decode_plan(n, n_heads, n_kv_heads, head_dim, bound, mean, most) + (1,)


def several_waves_cut(n_seqs: int, n_heads: int, n_kv_heads: int, head_dim: int, max_len: int, mean_len: int = 0):
    """The cut of an untuned decode launch whose whole contexts four waves of a workgroup walk between them, merging in LDS, which leaves no
    ranges to merge by a launch of their own; or None, where ``decode_plan`` decides.  Launch and merge, replayed over eight
    caches in turn, the rule's ranges -> this, us:

    - contexts of at most 1,024 keys and 512 on average, at 220 / 500 keys: 13 heads on 13 of 80, 1 sequence 7.6 -> 5.2, 7.9 -> 6.7, 5 8.1 -> 5.8,
      9.1 -> 7.4, 16 9.2 -> 6.9, 12.9 -> 9.5, 32 (416 workgroups) 9.0 -> 8.9, 17.2 -> 17.1; 71 on 1 of 64, 8 sequences 7.9 -> 5.3, 8.7 -> 7.7, 64
      (320) 13.0 -> 8.0, 13.9 -> 12.4; 128 on 8 of 64, 32 sequences 11.2 -> 6.4, 13.6 -> 9.3, 64 (512) 8.9 -> 8.6, 16.7 -> 16.2.  Heads of 128 carry twice
      the sums through LDS: 32 on 8, 8 sequences (64) 8.7 -> 7.5, 9.7 -> 11.4, 16 (128) 9.6 -> 7.6, 12.9 -> 11.7, 32 12.1 -> 9.0, 21.2 -> 16.3.
    - of at most 1,024 and more than 512 on average, heads up to 80, where workgroups are about as many as compute units, at 900 keys: 208 workgroups
      (13 on 13 of 80, 16 sequences) 20.3 -> 15.2; 256 (32 on 8 of 64, 32 sequences) 20.4 -> 14.9, (128 on 8) 20.3 -> 14.9; 104 to 128, which
      the same count of sequences (``decode_key``) stands for, 11.9 -> 10.1 to 15.6 -> 11.1.  With 320 it is 14.9 -> 18.8, with 416 27.0 either way,
      with 40 8.9 -> 10.3; and up to 2,048 keys 128 to 160 lose (16.4 -> 18.4 at 1,500) where 208 to 256 win (26.5 -> 22.0), under one count."""
    key = decode_key(n_seqs, n_heads, n_kv_heads, head_dim, max_len, mean_len)
    return None if key in _active.decode_plans else _several_waves_rule(*key)


def _several_waves_rule(n: int, n_heads: int, n_kv_heads: int, head_dim: int, bound: int, mean: int):
    if ops.ATTN_FORCE_SPLIT or ops.ATTN_FORCE_TILES or bound > 1024 or not ops.load_library().pta_attn_decode_waves_ok(head_dim, 1, 4):
        return None
    groups = n * n_kv_heads * ((n_heads // n_kv_heads + 15) // 16)  # workgroups of the launch
    if mean <= 512:
        if groups > 320 or (head_dim > 80 and groups < 128):
            return None
    elif head_dim > 80 or not 192 <= groups <= 256:
        return None
    return (1, bound, 4)


def _shared_keys_rule(n: int, n_heads: int, n_kv_heads: int, head_dim: int, bound: int, mean: int):
    """The cut with keys shared through LDS where it is built (many heads on a KV head) and the launch walks keys
    enough to fill the chip with such workgroups, else None.  Measured with 71 heads on one KV head of 64, launch
    and merge after a flush of the caches, against the best cut of one-wave workgroups: 8 sequences of 1,100 keys
    11.4 against 9.8 us; 32 of 1,100 10.3 against 15.4; 64 of 2,100 14.8 against 26.0; 8 of 16,384 19.8 against
    24.8; 32 of 16,384 45.6 against 49.8.  Ranges of 256 keys up to 100 k keys in all, 512 up to 300 k, then 1,024."""
    if ops.ATTN_FORCE_SPLIT or ops.ATTN_FORCE_TILES or not ops.attn_decode_shared_ok(head_dim, n_heads // n_kv_heads):
        return None
    keys = n * n_kv_heads * mean
    if keys < 20_000:
        return None
    size = 256 if keys <= 100_000 else 512 if keys <= 300_000 else 1024
    while size < bound and ((bound + size - 1) // size > 1024 or n * ((bound + size - 1) // size) > 65535):
        size *= 2  # the launch's limits: ranges of a sequence, and sequences x ranges
    return (1, min(size, bound), ops.SHARED_KEYS)


_decode_keys_seen: set = set()  # what decode launches asked ``decode_plan`` for while timing was on
_decode_keys_late: set = set()  # of those, where attention went in the launch of the products behind it (``late_waves``)


def note_decode_launch(n_seqs: int, n_heads: int, n_kv_heads: int, head_dim: int, max_len: int, mean_len: int = 0, late: bool = False) -> None:
    """While timing is on: remember that a decode launch of this shape ran, for ``CausalLM.tune`` to time its cuts."""
    if may_time():
        key = decode_key(n_seqs, n_heads, n_kv_heads, head_dim, max_len, mean_len)
        _decode_keys_seen.add(key)
        (_decode_keys_late.add if late else _decode_keys_late.discard)(key)


def take_decode_keys() -> list:
    """The (batch, head shape, context) counts of the decode launches since the last call, while timing was on."""
    keys = sorted(_decode_keys_seen)
    _decode_keys_seen.clear()
    return keys


def decode_plan_candidates(key) -> list:
    """Cuts of the decode launch that ``key`` counts, first the one that runs where none is fixed
    (``several_waves_cut``'s, else ``decode_plan``'s): the rules', the one-wave rule's neighbours,
    workgroups of four and eight waves over the whole context and over ranges of 512 and 1,024 keys, and, where
    they are built, workgroups that share their keys over ranges of 256 to 1,024 keys and the whole context.  A workgroup of several waves needs no second launch when it walks the whole context, but all its keys
    pass through one compute unit; which wins depends on how many sequences and KV heads there are to fill the
    chip.  Timed alone after a flush of the caches, these cuts rank differently than inside a step (the rule's
    cut at 64 sequences, 8 KV heads of 64 and 1,100 keys: 42 us alone, 31 us in a step, where a cut with four
    waves takes 34 us both times), so the caller times whole steps with each (``CausalLM.tune``)."""
    n, nh, nkv, d, bound, mean = key
    lib = ops.load_library()
    groups = (nh // nkv + 15) // 16
    most = min(groups, int(lib.pta_attn_decode_max_tiles(d)))
    rule = _decode_plan(n, nh, nkv, d, bound, mean, most) + (1,)
    # what runs where nothing was timed comes first: the caller measures the others against it
    late = (1, bound, 4) if tuple(key) in _decode_keys_late else None
    cuts = [c for c in dict.fromkeys((late, _several_waves_rule(*key), _shared_keys_rule(*key), rule)) if c is not None]
    want = [(rule[0], rule[1] * 2, 1), (rule[0], rule[1] // 2, 1), (max(1, rule[0] - 1), rule[1], 1),
            (min(most, rule[0] + 1), rule[1], 1)]
    want += [(t, size, w) for t in (1, min(2, most)) for w in (4, 8) for size in (bound, 1024, 512)]
    for t, size, w in want:
        size = min(size, bound)
        splits = (bound + size - 1) // size
        if (size < ops.ATTN_SPLIT_KEYS or size % 64 or size // w < 64 or splits > 1024 or n * splits > 65535 or (t, size, w) in cuts
                or not lib.pta_attn_decode_waves_ok(d, t, w)):
            continue
        cuts.append((t, size, w))
    if ops.attn_decode_shared_ok(d, nh // nkv):
        for size in (256, 512, 1024, bound):
            cut = (1, min(size, bound), ops.SHARED_KEYS)
            splits = (bound + cut[1] - 1) // cut[1]
            if cut not in cuts and splits <= 1024 and n * splits <= 65535:
                cuts.append(cut)
    return cuts


def context_lengths(longest: int, mean: int, n: int) -> list:
    """Lengths of ``n`` sequences whose longest and mean are given, for timing a step: all equal where the two are, spread evenly
    from next to nothing to the longest where the longest is twice the mean, more of them short beyond that, in no order.  How
    unequal they are and that they do not lie sorted decides between cuts: 16 sequences of 128 to 4,096 keys (32 heads on 8
    of 128, 60 layers) take 7.55 ms a step with one wave on 1,024 keys and 7.86 with four on 512, while with one sequence of
    4,096 and the others of 2,100 the second is the faster one (7.64 against 7.69), and with lengths sorted too (7.46, 7.56)."""
    longest, n = max(1, int(longest)), int(n)
    mean = max(1, min(int(mean), longest))
    bend = longest / mean - 1.0  # the mean of u^bend over 0..1 is mean / longest
    lens = [longest] + [min(longest, max(1, round(longest * ((n - 1 - i - 0.5) / (n - 1)) ** bend))) for i in range(n - 1)]
    left = max(mean * n, longest + n - 1) - sum(lens)  # the mean exactly: what is left over is shared out, within 1 to the longest
    while left:
        room = [i for i in range(1, n) if (lens[i] < longest if left > 0 else lens[i] > 1)]
        if not room:
            break
        each = max(1, abs(left) // len(room))
        for i in room[:abs(left)]:
            new = min(longest, lens[i] + each) if left > 0 else max(1, lens[i] - each)
            left -= new - lens[i]
            lens[i] = new
    return [lens[i] for i in sorted(range(n), key=lambda i: i * 0.6180339887498949 % 1.0)]


def set_decode_plan(key, cut=None) -> None:
    """Fix the cut of the decode launches that ``key`` counts (None: back to the rule)."""
    _note_change()
    if cut is None:
        _active.decode_plans.pop(tuple(key), None)
    else:
        _active.decode_plans[tuple(key)] = tuple(int(v) for v in cut)


# ---- when choices are timed -----------------------------------------------------------------------------
TUNE_LIVE = os.environ.get("PTA_TUNE", "0") == "1"


class live_tuning:
    """Context in which choices that have no entry in the tuning table yet are timed at first use."""

    def __enter__(self):
        global TUNE_LIVE
        self._old, TUNE_LIVE = TUNE_LIVE, True
        return self

    def __exit__(self, *exc):
        global TUNE_LIVE
        TUNE_LIVE = self._old
        _note_change()
        return False


def may_time() -> bool:
    return TUNE_LIVE and not torch.cuda.is_current_stream_capturing()


SKINNY_MAX_ROWS = 64
# rows up to which the decode batch kernel (x shared through LDS, K split over workgroups) stands in for the
# vendor library's product, whose choices for 65 to 128 rows leave most of the chip idle (K = 4,544 with N =
# 4,672 and 18,176 in one product of 128 rows: 151 us, 1.4 TB/s of weights)
SPLITK_MAX_ROWS = int(os.environ.get("PTA_SPLITK_MAX_ROWS", "256"))
SPLITK_MARGIN = float(os.environ.get("PTA_SPLITK_MARGIN", "0.95"))
SPLITK_SURE_ROWS = 128  # up to here the kernel won at every shape measured; beyond, by the weight's own timing


_flush = None  # half a gigabyte that is read between timed runs; held only while timing is on (``release_flush``)


def release_flush() -> None:
    global _flush
    _flush = None


def time_ways_cold(ways, device, rounds: int = 3):
    """Milliseconds of each of ``ways`` (callables), the fastest of ``rounds`` runs each, taken in turn; before
    every run half a gigabyte is read, so that the weights come from memory as they do in a model (timed back
    to back, a product finds its matrix in the memory-side cache and every way looks alike).  Read, not
    written: after half a gigabyte of writes the caches are full of lines that must go back to memory before
    anything else comes in, which no step of a model leaves behind, and a kernel that streams from memory then
    measures at little more than half its speed (decode attention over 144 MB of keys and values: 55 us after
    writes, 31 us in a step)."""
    global _flush
    if _flush is None or _flush.device != device:
        _flush = torch.zeros(128 * 1024 * 1024, dtype=torch.float32, device=device)
    flush = _flush
    best = [float("inf")] * len(ways)
    for run in ways:  # plans are made and the library set up before anything is timed
        run()
    for _ in range(rounds):
        for i, run in enumerate(ways):
            flush.sum()
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            run()
            end.record()
            end.synchronize()
            best[i] = min(best[i], start.elapsed_time(end))
    return best


def splitk_row_limit(*ws: torch.Tensor) -> int:
    """Rows up to which the decode batch kernel is the faster way to the product with ``w`` (or, for two weights, to
    the two products of a pair launch).  Up to 128 rows it always was (one chunk of rows per workgroup); with two
    chunks it depends on how well the product of many rows (``ops.mm_rows``) does at the shape, so both are timed once
    per shape at 192 and 256 rows, when timing is on; without an entry the kernel stops at 128 rows."""
    if SPLITK_MAX_ROWS <= SPLITK_SURE_ROWS:
        return SPLITK_MAX_ROWS
    key = tuple(tuple(w.shape) for w in ws)
    limit = _active.splitk_rows.get(key)
    if limit is None:
        if not may_time():
            return SPLITK_SURE_ROWS
        dev = ws[0].device
        xs = [torch.randn((256, w.shape[1]), dtype=torch.float32, device=dev).to(torch.bfloat16) for w in ws]
        limit = SPLITK_SURE_ROWS
        for rows in (192, 256):
            if rows > SPLITK_MAX_ROWS:
                break
            xr = [x[:rows] for x in xs]

            def kernel():
                if len(ws) == 1:
                    ops.gemm_splitk_bf16(xr[0], ws[0])
                else:
                    ops.gemm_splitk_pair_bf16(xr[0], ws[0], xr[1], ws[1])

            def product():
                for x, w in zip(xr, ws):
                    ops.mm_rows(x, w)

            best = time_ways_cold((kernel, product), dev)
            if best[0] < SPLITK_MARGIN * best[1]:
                limit = rows
            else:
                break
        _active.splitk_rows[key] = limit
    return limit


def splitk_rows_ok(x: torch.Tensor, *ws: torch.Tensor) -> bool:
    return x.shape[0] <= SPLITK_SURE_ROWS or x.shape[0] <= splitk_row_limit(*ws)


# ---- the vendor library's product for many rows, cut along M where that is faster -----------------------
# The library picks a kernel per (M, N, K) from a table, and on this hardware its choices are uneven in M:
# with K = 4,544 and N = 18,176, 2,048 rows take longer than 2,304, and 4,096 rows of the product with the
# transposed shape almost as long as 8,192.  So, when timing is on, the product is timed once per weight shape at
# a ladder of row counts, and a product of M rows then runs as the cheapest sequence of those pieces (each written
# straight into its rows of the result); without an entry it runs whole.  PTA_MM_CHUNKS=0 switches this off.
MM_LADDER = (256, 512, 768, 1024, 1536, 2048, 3072, 4096, 6144, 8192)
MM_CHUNKS = os.environ.get("PTA_MM_CHUNKS", "1") != "0"
MM_JOIN = os.environ.get("PTA_MM_JOIN", "1") != "0"  # one product for two matrices of one input where it is faster


def mm_measure(x: torch.Tensor, w: torch.Tensor, rows: int, out: torch.Tensor) -> float:
    """Microseconds of ``x[:rows] @ w.T``: the fastest of five runs, each timed on its own (a mean over two runs
    right after the library's set-up misjudged products by a tenth, enough to choose the slower plan)."""
    torch.mm(x[:rows], w.t(), out=out[:rows])  # the library's first call of a shape sets it up
    best = float("inf")
    for _ in range(5):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        torch.mm(x[:rows], w.t(), out=out[:rows])
        end.record()
        end.synchronize()
        best = min(best, start.elapsed_time(end) * 1e3)
    return best


def mm_plan(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor):
    M, (N, K) = x.shape[0], w.shape
    bucket = (M + 63) // 64  # row counts within 64 of each other share a plan: one timing of the whole product
    plan = _active.mm_plans.get((N, K, bucket))
    if plan is not None:
        return plan[:-1] + [M - sum(plan[:-1])]
    if not may_time():
        return [M]
    times = _active.mm_times.setdefault((N, K), {})
    for rows in MM_LADDER:
        if rows <= M and rows not in times:
            times[rows] = mm_measure(x, w, rows, out)
    whole = M <= MM_LADDER[-1]  # beyond the ladder the product always runs in pieces: timing it whole costs too much
    if whole and M not in times:
        times[M] = mm_measure(x, w, M, out)  # the product as it is
    # cheapest way to cover M rows with pieces of the ladder; what is left over rides on the last piece
    units, rest = divmod(M, 256)
    best = [(0.0, [])] + [None] * units
    for u in range(1, units + 1):
        for rows in MM_LADDER:
            k = rows // 256
            if k <= u and rows in times and best[u - k] is not None:
                cand = best[u - k][0] + times[rows]
                if best[u] is None or cand < best[u][0]:
                    best[u] = (cand, best[u - k][1] + [rows])
    cost, pieces = best[units]
    if rest:
        pieces = pieces[:-1] + [pieces[-1] + rest]
        cost *= M / (M - rest)
    plan = pieces if not whole or (len(pieces) > 1 and cost < 0.97 * times[M]) else [M]
    _active.mm_plans[(N, K, bucket)] = plan
    _active.mm_costs[(N, K, bucket)] = cost if plan is pieces else times[M]
    return plan


TILE_MARGIN = 0.98  # a way replaces the rule's only if it is faster by more than two runs of one way differ


def tile_pays(x: torch.Tensor, w: torch.Tensor, bias=None, act=None, add1=None, add2=None) -> bool:
    """Whether ``act(x @ w.T + bias) + add1 + add2`` of many rows runs in the hand-written kernel, which can take it, or through the
    library's product in the pieces of ``mm_plan``.  When timing is on, both are timed to their end once per shape and kind
    of epilogue (the hand-written kernel's own, a pass behind the library's); without an entry pieces that were timed for the
    shape hold (a table from before there was this choice), and else the rule (``ops.gemm_tile_rule``)."""
    M, (N, K) = x.shape[0], w.shape
    if not (_active.mm_tiles or _active.mm_plans or TUNE_LIVE):  # nothing was timed: steps launched directly are bound by the host
        return ops.gemm_tile_rule(M, N, K)
    bucket = (M + 63) // 64
    key = (N, K, bucket, ops.ACT_CODES[act], int(bias is not None), (add1 is not None) + (add2 is not None))
    pays = _active.mm_tiles.get(key)
    if pays is not None:
        return pays
    rule = ops.gemm_tile_rule(M, N, K)
    if not may_time():
        return rule and not (MM_CHUNKS and (N, K, bucket) in _active.mm_plans)
    rest = (bias, act, add1, add2)
    tile, library = time_ways_cold((lambda: ops.tile_rows(x, w, *rest), lambda: ops.library_rows(x, w, *rest)), x.device)
    pays = not library < TILE_MARGIN * tile if rule else tile < TILE_MARGIN * library
    _active.mm_tiles[key] = pays
    return pays


def joined_mm_pays(x: torch.Tensor, joined: torch.Tensor, n_first: int, bias1=None, act1=None, bias2=None, act2=None) -> bool:
    """Whether the products with the first ``n_first`` rows of ``joined`` and with the rest, each with its bias and
    activation, are faster as one product (``ops.joined_rows``: bias and activation are passes behind it) than on their own
    (``ops.mm_rows``).  How evenly the tiles of each fill the chip decides (and where it is the library's product,
    its kernel choice), so both ways are timed to their end once per shape when timing is on; without an entry the two
    stay apart."""
    M, (N, K) = x.shape[0], joined.shape
    if not MM_JOIN or not MM_CHUNKS or M < 512:
        return False
    bucket = (M + 63) // 64
    key = bare = (n_first, N - n_first, K, bucket)
    if not (bias1 is None and act1 is None and bias2 is None and act2 is None):
        key += (ops.ACT_CODES[act1], int(bias1 is not None), ops.ACT_CODES[act2], int(bias2 is not None))
    if key not in _active.mm_joined:
        if not may_time():
            return _active.mm_joined.get(bare, False)  # (a table from before the epilogues counted says it by the shape alone)
        first, rest = joined[:n_first], joined[n_first:]
        ways = (lambda: ops.joined_rows(x, joined, n_first, bias1, act1, bias2, act2),
                lambda: (ops.mm_rows(x, first, bias1, act1), ops.mm_rows(x, rest, bias2, act2)))
        best = [float("inf"), float("inf")]
        for run in ways:  # plans are made and the library set up before anything is timed
            run()
        for _ in range(4):  # the two ways in turn, each run timed on its own; the fastest of each counts
            for i, run in enumerate(ways):
                start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                start.record()
                run()
                end.record()
                end.synchronize()
                best[i] = min(best[i], start.elapsed_time(end))
        _active.mm_joined[key] = best[0] < 0.98 * best[1]
    return _active.mm_joined[key]


# Ranges of K for the pairs of a shape: the kernel library's rule gives a choice per class of rows; when timing is on,
# its neighbours are timed once per shape, with cold caches, at rows of the class, and one that is at least 3 % faster is kept for
# every later launch of the class (PTA_PAIR_TUNE=0 switches this off).
PAIR_TUNE = os.environ.get("PTA_PAIR_TUNE", "1") != "0"
PAIR_TUNE_MARGIN = 0.97
PAIR_TUNE_ROWS = int(os.environ.get("PTA_PAIR_TUNE_ROWS", "64"))  # the larger of the two counts timed for 33 to 64 rows


def pick_way(times, margin: float) -> int:
    """The way to take, by times[count of rows][way]: the first, which is the rule's, unless another is no slower at any count
    and faster by the margin over them together; then the fastest of those."""
    total = [sum(t[i] for t in times) for i in range(len(times[0]))]
    ok = [i for i in range(1, len(total)) if total[i] < margin * total[0] and all(t[i] <= t[0] for t in times)]
    return min(ok, key=lambda i: total[i]) if ok else 0


RIDE_KEYS = 150  # of every sequence, where a pair is timed with the attention that it may carry


def ride_gain(copies, late, x1: torch.Tensor, stream: torch.Tensor, norm_w: torch.Tensor) -> float:
    """Milliseconds that the pair's launch saves by carrying a decode step's attention (``ops.gemm_splitk_pair_attn``), against attention in
    a launch of its own, with the ranges that are fixed for the pair: 0 where it does not carry it.  ``copies``: pairs of matrices, each read from memory;
    ``late``: what the step that is timed would hand over (an ``ops.LateAttention``), whose heads are taken with contexts of ``RIDE_KEYS``
    for as many sequences as ``x1`` has rows.  The norm of ``stream`` and both products follows either way.  Replays of captured
    launches are timed, because the host takes longer for two launches than a small pair does."""
    rows, (nh, d), nkv = x1.shape[0], late.q.shape[1:], late.k_pool.shape[1]
    (N1, K1), (N2, K2) = copies[0][0].shape, copies[0][1].shape
    waves = late_waves(rows, nh, nkv, d, RIDE_KEYS, RIDE_KEYS) if rows <= ops.LATE_MOST_ROWS else 0
    if not waves or not ops.load_library().pta_gemm_splitk_pair_attn_ok(N1, K1, N2, K2, rows, nh, nkv, d):
        return 0.0
    pages = (RIDE_KEYS + 63) // 64
    draw = lambda *shape: torch.randn(shape, device=x1.device).to(torch.bfloat16)
    count = lambda *a: torch.arange(*a, dtype=torch.int32, device=x1.device)
    start = torch.full((rows,), RIDE_KEYS - 1, dtype=torch.int32, device=x1.device)
    ctx = copy.copy(late.ctx)
    ctx.n_seqs = ctx.n_tokens = rows
    ctx.token_seq, ctx.cu_tokens, ctx.token_pos, ctx.seq_start = count(rows), count(rows + 1), start, start
    ctx.new_tokens, ctx.is_decode, ctx.max_len, ctx.mean_len, ctx.extras = [1] * rows, True, RIDE_KEYS, RIDE_KEYS, {}
    trial = ops.LateAttention(draw(rows, nh, d), draw(rows * pages, nkv, 64, d), draw(rows * pages, nkv, d, 64), count(rows * pages).view(rows, pages),
                              ctx, late.slopes, late.scale, waves=waves, **late.how)
    if not ops.late_attention_pays(trial, *copies[0]):
        return 0.0
    parts = [torch.empty((p, rows, N), dtype=torch.float32, device=x1.device)
             for p, N in zip(ops.gemm_splitk_pair_parts(N1, K1, N2, K2, rows), (N1, N2))]

    def apart(a, b):
        trial.run()
        ops._call("pta_gemm_splitk_pair_bf16", ops._ptr(parts[0]), ops._ptr(x1), ops._ptr(a), int(N1), int(K1), ops._ptr(parts[1]),
                  ops._ptr(trial.out), ops._ptr(b), int(N2), int(K2), rows, ops._stream())
        return parts

    def together(a, b):
        return ops.gemm_splitk_pair_attn(x1, a, trial, b)

    def ms(way) -> float:
        def run():
            ctx.extras.clear()  # (marks that are clear when a launch starts are cleared in the capture)
            for a, b in copies:
                first, second = way(a, b)
                ops.layernorm_sum([(second, None), (first, None), stream], N1, w=norm_w, b=norm_w, eps=1e-5)

        run()
        torch.cuda.synchronize(x1.device)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            run()
        best = float("inf")
        for _ in range(6):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            graph.replay()
            end.record()
            end.synchronize()
            best = min(best, begin.elapsed_time(end) / len(copies))
        return best

    return ms(apart) - ms(together)


def tune_pair_parts(w1: torch.Tensor, w2: torch.Tensor) -> None:
    """``tune_pair_carrying`` of a pair whose launch carries nothing else."""
    tune_pair_carrying(w1, w2, None)


def tune_pair_carrying(w1: torch.Tensor, w2: torch.Tensor, late) -> None:
    """Once per pair of shapes, while timing is on: the pair launch with the ranges of K that the rule has for the rows, and with
    neighbours of them, with cold caches; ``pick_way`` says which is kept.  Up to 32 rows are timed at 8 and 32; 33 to 64 rows,
    where they have ranges of their own, at 40 and 64, and with workgroups of 128 rows of W (which load the activations half as
    often, have half as many workgroups and so want more ranges); those are timed at 128 rows too, with the ranges of few rows.  Then, at 8, 32, 64 and 128 rows (one count per class of
    rows), the launch with stationary activations is timed against the winner with one to six ranges of the shorter K
    (and as many times more of the longer): whichever of the two the rule takes for the class stays unless it is beaten by 2 %.
    All with what reads the partial sums behind the launch (the norm that adds them, where the two products have one width;
    else a charge for the ranges' bytes).  Where the step's attention may go in the pair's launch (``late``, an ``ops.LateAttention``), a way that
    cannot carry it (six waves, stationary activations) is charged what that saves (``ride_gain``).  ``TuningTable.pair_parts`` and
    ``pair_stationary`` keep what is in use.

    The rule's choice for the class is what has to be beaten, at rows of the class, because ranges that are 14 % faster at 64 rows may be
    slower at 8 (4,544 x 4,544 + 4,544 x 18,176, where a single timing at 64 rows chose for all: a step of 7B layers 3.07 -> 3.17 ms at 8
    sequences, 3.61 -> 3.68 at 32)."""
    key = (tuple(w1.shape), tuple(w2.shape))
    if not PAIR_TUNE or key in _active.pair_parts or not may_time():
        return
    lib = ops.load_library()
    (N1, K1), (N2, K2) = w1.shape, w2.shape
    shapes = (int(N1), int(K1), int(N2), int(K2))
    class_rows = (8, 32, 64, 128)
    rules = [ops.gemm_splitk_pair_way(*shapes, rows) for rows in class_rows]  # nothing is fixed for the shapes yet
    few, middle = rules[0], rules[2] if rules[2][2] != 3 else None
    fix = lambda c: lib.pta_gemm_splitk_pair_fix(*shapes, int(c[0]), int(c[1]), int(c[2]))
    forget = lambda: lib.pta_gemm_splitk_pair_fix(*shapes, 0, 0, 1)
    fix_st = lambda cls, c: lib.pta_gemm_splitk_pair_fix_stationary(*shapes, int(cls), int(c[0]), int(c[1]))
    for cls in range(len(class_rows)):
        fix_st(cls, (0, 0))  # the launches timed first are the staged kernel's
    near = lambda a0, b0: [(a, b, 1) for a in range(max(1, a0 - 1), a0 + 3) for b in range(max(1, b0 - 2), b0 + 3)]
    tall = lambda a0, b0: [(a, b, 2) for a in sorted({max(1, a0 - 1), a0, a0 + 1, max(1, 2 * a0 - 1), 2 * a0, 2 * a0 + 1})
                           for b in sorted({max(1, b0 - 1), b0, b0 + 1, max(1, 2 * b0 - 1), 2 * b0, 2 * b0 + 1})]
    six = lambda a0, b0: [(a, b, 4) for a in range(max(1, a0 - 1), a0 + 2) for b in range(max(1, b0 - 1), b0 + 2)]
    ways = lambda rule, others: [rule] + [c for c in dict.fromkeys(others) if c != rule and fix(c) == 0]  # those that the kernel takes
    few_ways = ways(few, near(*few[:2]))
    middle_ways = ways(middle, near(*middle[:2]) + near(*few[:2]) + tall(*middle[:2]) + tall(*few[:2]) + six(*middle[:2])) if middle else []
    larger = min(64, max(41, PAIR_TUNE_ROWS))
    counts = {rows: [torch.randn((rows, K), dtype=torch.float32, device=w1.device).to(torch.bfloat16) for K in (K1, K2)]
              for rows in sorted({*class_rows, 40, larger})}
    xs_bf16 = {rows: torch.zeros((rows, N1), dtype=torch.bfloat16, device=w1.device) for rows in counts}
    kmin = min(K1, K2)
    f1, f2 = max(1, (K1 + kmin // 2) // kmin), max(1, (K2 + kmin // 2) // kmin)
    st_cands = [(b * f1, b * f2) for b in (1, 2, 3, 4, 6) if b * f1 <= 16 and b * f2 <= 16]
    st_cands = [c for c in dict.fromkeys([r[:2] for r in rules if r[2] == 3] + st_cands) if fix_st(0, c) == 0]
    fix_st(0, (0, 0))
    most = [max([c[i] for c in few_ways + middle_ways] + [c[i] for c in st_cands] + [16]) for i in (0, 1)]
    parts = [torch.empty((most[i], 128, N), dtype=torch.float32, device=w1.device) for i, N in enumerate((N1, N2))]
    # A launch is timed over several copies of the matrices in turn (more bytes than the memory-side cache holds),
    # back to back between two events: every launch reads its matrices from memory, as in a model, and no gap of
    # the host's lies inside the timed span.
    copy_bytes = (w1.numel() + w2.numel()) * 2
    n_copies = max(2, min(6, int(640e6 // copy_bytes) + 1))
    copies = [(w1, w2)] + [(w1.clone(), w2.clone()) for _ in range(n_copies - 1)]

    # Two products of the same width are a block's last ones, and what reads their partial sums next is the norm
    # that adds them: it is launched behind every timed launch, so that a launch pays for
    # the ranges it leaves to be added and for how it leaves them (all at once at its end, or as it goes).
    norm_w = (torch.ones(N1, dtype=torch.float32, device=w1.device)
              if N1 == N2 and ops.layernorm_sum_ok(N1) and os.environ.get("PTA_PAIR_TUNE_READER", "1") != "0" else None)

    def read_sums(c, rows):
        views = [parts[i].view(-1)[:int(c[i]) * rows * N].view(int(c[i]), rows, N) for i, N in enumerate((N1, N2))]
        ops.layernorm_sum([(views[1], None), (views[0], None), xs_bf16[rows]], N1, w=norm_w, b=norm_w, eps=1e-5)

    def timed_ways(chosen, rows, fix, rounds=4):
        """Milliseconds of a launch and of reading its sums, for each of the ways (ranges, ranges, ..) that ``fix`` sets."""
        best = [float("inf")] * len(chosen)
        for r in range(rounds + 1):  # the first round warms up
            for j, c in enumerate(chosen):
                fix(c)
                start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                start.record()
                for a, b in copies:
                    ops._call("pta_gemm_splitk_pair_bf16", ops._ptr(parts[0]), ops._ptr(counts[rows][0]), ops._ptr(a), int(N1), int(K1),
                          ops._ptr(parts[1]), ops._ptr(counts[rows][1]), ops._ptr(b), int(N2), int(K2), rows, ops._stream())
                    if norm_w is not None:
                        read_sums(c, rows)
                end.record()
                end.synchronize()
                if r > 0:
                    best[j] = min(best[j], start.elapsed_time(end) / len(copies))
        # (what reads partial sums afterwards takes some 8 TB/s worth of them)
        return best if norm_w is not None else [t + (c[0] * N1 + c[1] * N2) * rows * 4 / 8e12 * 1e3 for t, c in zip(best, chosen)]

    say = (lambda text: print(f"[pta tune] pair {key}: {text}", flush=True)) if os.environ.get("PTA_TUNE_VERBOSE") else (lambda text: None)

    def saved(rows):  # by the launch that carries attention, with what is fixed now
        if late is None or norm_w is None or ops._timing is not None:
            return 0.0
        gain = ride_gain(copies, late, counts[rows][0], xs_bf16[rows], norm_w)
        if gain:
            say(f"at {rows} rows: attention in the launch saves {gain * 1e3:.1f} us")
        return gain

    def choose(found, label, rows):
        times = [timed_ways(found, n, fix) for n in rows]
        carry = [c[2] != 4 for c in found]
        if any(carry) and not all(carry):
            for n, t in zip(rows, times):
                fix(found[min((j for j, c in enumerate(carry) if c), key=lambda j: t[j])])
                gain = saved(n)
                t[:] = [v if c else v + gain for v, c in zip(t, carry)]
        i = pick_way(times, PAIR_TUNE_MARGIN)
        show = lambda j: f"{found[j]} " + " / ".join(f"{t[j] * 1e3:.1f}" for t in times)
        say(f"{label}: rule {show(0)} us; fastest " + ", ".join(show(j) for j in sorted(range(len(found)), key=lambda j: sum(t[j] for t in times))[:5]) +
            f" -> {found[i]}")
        return found[i]

    chosen_st = []
    try:
        a, b, _ = choose(few_ways, "8 / 32 rows", (8, 32))
        cut = choose([(a, b, 1), (a, b, 2)], "128 rows", (128,))  # (the tile height counts beyond 32 rows)
        if middle:
            cut = cut + choose(middle_ways, f"40 / {larger} rows", (40, larger))
        _fix_pair(*key, cut)
        # the launch with stationary activations against that choice, per class of rows
        for cls, rows in enumerate(class_rows):
            # the fewest ranges among those within 1.5 % of the fastest: what separates them is less than a box
            # varies, and fewer ranges leave whatever reads them next less to read
            staged = ops.gemm_splitk_pair_parts(*shapes, rows)
            t_staged = timed_ways([staged], rows, lambda c: fix_st(cls, (0, 0)))[0]
            gain = saved(rows) if st_cands else 0.0
            t_st = timed_ways(st_cands, rows, lambda c: fix_st(cls, c)) if st_cands else []
            best = min((i for i in range(len(st_cands)) if t_st[i] <= 1.015 * min(t_st)), key=lambda i: st_cands[i]) if st_cands else -1
            found = [((0, 0), t_staged)] + ([(st_cands[best], t_st[best] + gain)] if best >= 0 else [])
            if rules[cls][2] == 3:  # the rule's ranges first
                found.insert(0, (rules[cls][:2], t_st[st_cands.index(rules[cls][:2])] + gain))
            keep = found[pick_way([[t for _, t in found]], 0.98)][0]
            chosen_st.append(keep)
            fix_st(cls, (0, 0))
            say(f"at {rows} rows: staged {t_staged * 1e3:.1f} us; stationary " + ", ".join(f"{c} {t * 1e3:.1f}" for c, t in zip(st_cands, t_st)) +
                f"; rule {rules[cls]} -> {keep}")
    except BaseException:
        forget()
        fix_st(-1, (0, 0))
        raise
    for cls, c in enumerate(chosen_st):
        fix_st(cls, c)
    _active.pair_parts[key] = cut
    _active.pair_stationary[key] = tuple(chosen_st)


def gemm_splitk_pair_parts_rule(N1: int, K1: int, N2: int, K2: int):
    """The ranges of K that the kernel library's own rule gives a pair, whatever has been fixed for the shape."""
    lib = ops.load_library()
    kept = _active.pair_parts.get(((int(N1), int(K1)), (int(N2), int(K2))))
    lib.pta_gemm_splitk_pair_fix(int(N1), int(K1), int(N2), int(K2), 0, 0, 1)
    rule = ops.gemm_splitk_pair_parts(N1, K1, N2, K2)
    if kept is not None:
        _fix_pair((N1, K1), (N2, K2), kept)
    return rule


# Elements of both matrices of a pair launch up to which it beats the two products on their own beyond 48 rows.
# Measured in whole decode steps: pairs of 104 M elements (K = 4,544, N = 4,672 + 18,176) and of 92 M (K = 4,096, N
# = 6,144 + 16,384) win at every row count; a pair of 344 M (K = 8,192, N = 9,216 + 32,768) wins up to 48 rows (32
# rows: 20.8 against 23.0 ms a step) and loses beyond them to the vendor library's product for the longer matrix
# (64 rows: 24.3 against 23.3 ms).
PAIR_MAX_WEIGHTS = 160 * 1024 * 1024
PAIR_SURE_ROWS = 48


def pair_launch_pays(rows: int, w1: torch.Tensor, w2: torch.Tensor) -> bool:
    """Whether two products of ``rows`` rows (17 and more) run as one launch of the decode batch kernels."""
    return rows <= PAIR_SURE_ROWS or w1.numel() + w2.numel() <= PAIR_MAX_WEIGHTS
