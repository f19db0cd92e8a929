"""The prefill launches' split of their work, as a model of the host plan and the device ranges.

A prefill call's row groups (256 rows) hold stages of 64 keys; each launch gives every workgroup a
contiguous range of the stages of all row groups, weighted by what starting one costs.  Whatever the
shapes and the actual lengths (the plan is made for the longest sequence), every stage of every
row group must belong to exactly one workgroup, the segments of a row group must fit its statistics,
and every part slot must be its segment's own and lie inside the workspace.  Calls over short
contexts take whole row groups of 128 rows instead.
"""
import random

import pytest

from specdec_amd import _native

ROWS, SHORT_ROWS, STAGE, SEG, MIN, CUS = 256, 128, 64, 6, 3, 256
SYNC_PART, DESC, MAX_GROUPS = 8 << 20, (1 << 14) * 8, 1 << 14


def cdiv(a, b):
    return -(-a // b)


def stages(i, s, g, t, rows=ROWS):
    last = min(s - 1, (rows * (i + 1) - 1) // g)
    return max(1, (t - s + last + STAGE) // STAGE if t - s + last + STAGE > 0 else 0)


def short(groups, r, s, g, d, t):
    """Whether the call takes whole row groups of 128 rows."""
    nrg = cdiv(r, SHORT_ROWS)
    n = groups * nrg
    most = (6 if n < 4 else 8 if n < 32 else 10) if d == 128 else (9 if n < 4 else 11 if n < 32 else 12)
    return stages(nrg - 1, s, g, t, SHORT_ROWS) <= most


def plan(groups, r, s, g, d, t):
    """plan_prefill of csrc/sdv_attn.hip: (workspace bytes, w1, w2, min1, split, slots, dense)."""
    nbk = cdiv(t, 16)
    max_parts = min(64, max(1, nbk // 8))
    n128 = cdiv(r, 128)
    split = max(1, min(max_parts, (1536 if d == 128 else 1792) // (groups * n128)))
    budget = 512 if d == 128 else 768
    parts = max(1, min(min(max_parts, 8), budget // (groups * n128))) if groups * n128 <= (4096 * 64 * 16) // 8 else 1
    if parts > 1 and s % 128 == 0:
        for kstar in range(4, nbk + 4, 4):
            pk = [max(1, cdiv(max(0, cdiv(t - s + min(s, 128 * (k + 1)), 16)), kstar)) for k in range(s // 128)]
            if groups * g * sum(pk) <= budget and max(pk) <= 8:
                parts = max(pk) if max(pk) > 1 else parts
                break
    slot_bytes = cdiv(groups * n128 * parts * 128 * d * 4, 256) * 256 if parts > 1 else 0
    total = (_native.SYNC_BYTES + cdiv(groups * r * 8 * split, 256) * 256 + slot_bytes
             + groups * ((nbk + 1) // 2) * (d // 16) * 1024)
    nrg = cdiv(r, ROWS)
    u = groups * sum(SEG + stages(i, s, g, t) for i in range(nrg))
    slot_b = ROWS * d * 4
    slots = slot_bytes // slot_b
    have = slots + (SYNC_PART - DESC) // slot_b
    n = groups * nrg
    w2 = min(CUS, max(have // 2, have - n), cdiv(u, MIN))
    if short(groups, r, s, g, d, t):
        return total, 0, 0, MIN, split, slots, False, have
    if u >= 1 << 30 or nbk >= 1 << 22 or n > MAX_GROUPS or w2 < min(n, CUS):
        return total, 0, 0, MIN, split, slots, False, have
    w1, min1 = 0, MIN
    if split >= 2:
        w1 = min(CUS, cdiv(u, MIN))
        min1 = max(min1, cdiv(stages(nrg - 1, s, g, t) - 1, split - 1))
    return total, w1, w2, min1, split, slots, w2 + n <= have, have


def ranges(w, minper, wts):
    """Segments of every row group under w workgroups: [(first workgroup, [(stage lo, hi), ...])]."""
    u = sum(wts)
    per = max(cdiv(u, w), minper)
    segs = [[] for _ in wts]
    for wg in range(w):
        lo, hi = min(wg * per, u), min(min(wg * per, u) + per, u)
        start = 0
        for f, wt in enumerate(wts):
            if lo < start + wt and hi > start:
                slo, shi = max(lo - start - SEG, 0), min(hi - start, wt) - SEG
                if slo < shi:
                    segs[f].append((wg, slo, shi))
            start += wt
    return per, segs


def check(groups, b, kv, g, s, d, lens):
    r, tmax = g * s, max(lens)
    total, w1, w2, min1, split, slots, dense, have = plan(groups, r, s, g, d, tmax)
    nrg = cdiv(r, ROWS)
    if w2 == 0:
        return total, False
    lk = groups // b
    wts = [SEG + stages(i, s, g, t) for _ in range(lk) for t in lens for i in range(nrg)]
    for w, minper, first in ((w1, min1, True), (w2, MIN, False)):
        if w == 0:
            continue
        per, segs = ranges(w, minper, wts)
        start, ids = 0, set()
        for rgi, (wt, sg) in enumerate(zip(wts, segs)):
            assert [x[1] for x in sg] == [0] + [x[2] for x in sg[:-1]] and sg[-1][2] == wt - SEG, "stages covered once, in order"
            w0, n = (start + SEG) // per, (start + wt - 1) // per - (start + SEG) // per + 1
            assert [x[0] for x in sg] == list(range(w0, w0 + n)), "the segments are those of consecutive workgroups"
            if first:
                assert n <= split
            elif n > 1:
                for k in range(n):
                    slot = w0 + k + rgi if dense else 2 * (w0 + k) + (k == 0)
                    assert slot not in ids and 0 <= slot < have
                    ids.add(slot)
            start += wt
    return total, True


@pytest.mark.parametrize("seed", range(6))
def test_ranges_cover_every_stage_once(seed):
    rng = random.Random(seed)
    lib = _native.load()
    split = 0
    for _ in range(60):
        d, g = rng.choice([(128, 6), (64, 7)])
        kv, layers, b = rng.choice([1, 2]), rng.choice([1, 1, 2, 5]), rng.choice([1, 1, 2, 3, 9])
        s = int(2 ** rng.uniform(3.6, 11))
        s += (64 // g + 1 - s) if g * s <= 64 else 0
        tmax = max(s, int(2 ** rng.uniform(6, 15)))
        lens = [tmax] + [rng.randint(0, tmax) for _ in range(b - 1)]
        total, ok = check(layers * b * kv, b, kv, g, s, d, lens)
        split += ok
        assert lib.sdv_attention_workspace_size(layers, b, g * kv, kv, s, d, tmax) == total
    assert split > 20, "most of these calls split their row groups"


def test_large_calls_take_whole_row_groups():
    assert check(28 * 32 * 2, 32, 2, 6, 2048, 128, [8192] * 32)[1] is False
