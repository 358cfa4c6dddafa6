"""pd_native (csrc/pd_python.cpp) on the CPU: the split plans equal their models, and errors come back as the
Python exceptions that the operators document. The calls themselves are covered by every GPU test.
"""
import heapq
import math
import os
import random
import re

import numpy as np
import pytest
import torch

from mi50_vllm_lab_amd import kvcache, pth_dec
from mi50_vllm_lab_amd import vllm_shim as shim


def decode_model(nseg, window, hkv, lens, max_q, hq, cus=256):
    """vllm_shim.decode_splits' makespan model in numpy, for batches that are not sliced."""
    cap = max(1, min(64, nseg))
    n = len(lens)
    x = np.minimum(lens, window + max_q) if window > 0 else np.asarray(lens)
    tiles = (x + 31) // 32 + (x > 0)
    live = tiles > 0
    if not live.any():
        return 1
    best, best_t = cap, math.inf
    for s in sorted({1 << k for k in range(int(math.log2(cap)) + 1)} | {cap}):
        per = np.maximum(-(-tiles // s), 1)
        used = np.where(live, -(-tiles // per), 0)
        t = shim.SPLIT_FIXED_US + shim.SPLIT_TILE_US * -(-per // 4)
        span = max(hkv * float(np.sum(used * t + (s - used) * shim.SPLIT_EMPTY_US)) / cus, float(t[live].max()))
        span += shim.COMBINE_US_PER_MB * n * max_q * hq * s * shim.PARTIAL_ROW_BYTES / 1e6
        if span < best_t - 1e-9:
            best, best_t = s, span
    return best


@pytest.mark.parametrize("seed", range(8))
def test_decode_plan_equals_its_model(seed):
    r = random.Random(seed)
    for _ in range(200):
        n = r.randint(1, r.choice([3, 20, 130]))
        lens = np.array([r.choice([0, r.randint(1, 200000), r.randint(1, 3000)]) for _ in range(n)])
        nseg, window, hkv, max_q = r.choice([1, 2, 7, 16, 64, 128]), r.choice([-1, -1, 9000, 30000]), r.choice([1, 2, 4, 8]), r.choice([1, 2, 4])
        if shim.sliced_splits(window, max_q, 6, hkv, n, 256, min(64, nseg)):
            continue
        want = decode_model(nseg, window, hkv, lens, max_q, 6 * hkv)
        for given in (lens.tolist(), lens, torch.from_numpy(lens), torch.from_numpy(lens.astype(np.int32))):
            assert shim.decode_splits(nseg, window, hkv, n, "cpu", given, max_q) == want


def deal_model(lens, hkv, max_q, window, cus):
    """pd_native.deal_pays: the workgroups in order on the CU that is free first, against an equal share."""
    tiles = [-(-min(x, window + max_q if window > 0 else x) // 32) + 1 for x in lens if x > 0]
    free = [0] * max(1, cus // hkv)
    for t in tiles:
        at = free.index(min(free))
        free[at] += t + 12
    return max(free) > 1.15 * hkv * sum(t + 12 for t in tiles) / cus + 8


@pytest.mark.parametrize("seed", range(4))
def test_deal_rating_equals_its_model(seed):
    r = random.Random(seed)
    seen = set()
    for _ in range(150):
        n, top = r.randint(1, r.choice([20, 130, 400])), r.choice([100, 1500, 20000])
        lens = [r.choice([0, top, r.randint(1, top), top - r.randint(0, top // 8)]) for _ in range(n)] if r.random() < 0.5 else [top] * n
        hkv, max_q, window, cus = r.choice([1, 2, 3, 8]), r.choice([1, 4]), r.choice([-1, 900]), r.choice([1, 40, 256])
        want = deal_model(lens, hkv, max_q, window, cus)
        for given in (torch.tensor(lens), torch.tensor(lens, dtype=torch.int32)):
            assert pth_dec.native().deal_pays(given, n, hkv, max_q, window, cus) == want
        seen.add(want)
    assert seen == {False, True}


# sequences' keys (24 q / 4 kv heads, one token), us in one workgroup per sequence and kv head, us dealt
UNSPLIT_BATCHES = [([1024] * 128, 57.5, 59.9), ([64] * 128, 21.3, 25.9), ([512] * 256, 77.6, 82.3), ([256] * 512, 128.1, 144.9),
                   ([1024 - 32 * (i % 16) for i in range(128)], 49.7, 55.4), ([1000] * 65, 46.6, 37.4), ([2048] * 96, 100.3, 94.2),
                   ([8192] * 70, 316, 228), ([100 + 18 * (i * 37 % 160) for i in range(160)], None, 0)]


@pytest.mark.parametrize("lens,unsplit,dealt", UNSPLIT_BATCHES)
def test_unsplit_batches_are_launched_as_measured(lens, unsplit, dealt):
    batch = (64, -1, 4, len(lens), "cpu", lens, 1, 24)
    assert shim.decode_splits(*batch) == 1
    want = 2 if unsplit is None or dealt < unsplit else 1
    assert shim.launched_splits(1, *batch) == want
    assert shim.launched_splits(1, 2, *batch[1:]) == 1            # no segments for the deal
    assert shim.launched_splits(1, *batch[:5], None, 1, 24) == 1  # no lengths
    assert shim.launched_splits(4, *batch) == 4
    assert shim.launched_splits(1, *batch[:6], 8, 48) == 1        # more than 32 rows per kv head


@pytest.mark.parametrize("seed", range(8))
def test_prefill_plan_equals_its_model(seed):
    r = random.Random(seed)
    for _ in range(100):
        hkv = r.choice([1, 2, 4, 8])
        a = (r.randint(1, 4), r.choice([r.randint(1, 100), r.randint(1, 5000)]), hkv * r.choice([1, 4, 6, 8]), hkv,
             r.choice([0, r.randint(1, 2000), r.randint(1, 300000)]))
        bs = r.choice([1, 8, 16, 48, 1584])
        top = max(1, min(pth_dec.PREFILL_MAX_SPLITS, -(-a[4] // 32) // pth_dec.PREFILL_MIN_TILES_PER_SPLIT))
        counts = [s for s in range(1, top + 1) if s == 1 or a[0] * a[1] * a[2] * s * 1032 <= pth_dec.PREFILL_MAX_WORKSPACE]
        assert pth_dec.prefill_splits(*a, bs) == min(counts, key=lambda s: pth_dec.prefill_cost_us(*a, s, bs))


PLAN = open(os.path.join(os.path.dirname(pth_dec.__file__), "csrc", "pd_plan.hpp")).read()
TIMES = {e: [float(x) for x in re.search(r"constexpr FaTimes %s = \{(.*?)\}" % n, PLAN).group(1).split(",")]
         for e, n in ((False, "kFaTimes"), (True, "kFaTimesExact"))}
SEGMENT, MIN_SHARE, ALIGNED, SPARE, DEAL_US, MARGIN = (
    float(re.search(r"constexpr \w+ %s = ([\d.]+);" % n, PLAN).group(1))
    for n in ("kFaSegmentUnits", "kFaMinShare", "kFaAlignedPart", "kFaDealSpareUnits", "kFaDealFixedUs", "kFaDealMargin"))


def chunk_model(batch, sq, hq, hkv, keys, bs, exact, cus=256):
    """pd_native.plan_prefill for a chunk whose tokens are the last of `keys` keys: {split count: (us, kernel)}, the us of
    the dealt launch (None where it would cut the query tiles evenly), and the us of a split count in the order of its
    workgroups."""
    tile, wide, unit = TIMES[exact]
    g, tiles = hq // hkv, -(-keys // 32)
    tok = 192 // g
    qtiles = -(-sq // tok)
    items, wide_items, rows = qtiles * hkv * batch, -(-sq * g // 256) * hkv * batch, batch * sq * hq
    out = {}
    for s in range(1, max(1, min(64, tiles // 8)) + 1):
        if s > 1 and rows * s * 1032 > pth_dec.PREFILL_MAX_WORKSPACE:
            break
        per = -(-tiles // s)
        table = 2 * per if bs % 16 == 0 else -(-keys // bs)
        slow = 1.0 if table <= pth_dec.PREFILL_LDS_TABLE else pth_dec.PREFILL_GLOBAL_TABLE_FACTOR
        rounds, wide_rounds = -(-items * s // cus), -(-wide_items * s // cus)
        merge = pth_dec.PREFILL_US_MERGE_LAUNCH + pth_dec.PREFILL_US_PER_PARTIAL_MB * rows * s * 1032 / 1e6 if s > 1 else 0.0
        times = {192: rounds * (per * tile * slow + pth_dec.PREFILL_US_PER_WORKGROUP) + merge}
        if wide_rounds * wide < rounds * tile:
            times[256] = wide_rounds * (per * wide * slow + pth_dec.PREFILL_US_PER_WORKGROUP) + merge
        out[s] = min((t, k) for k, t in times.items())
    units = sum(-(-(max(0, keys - sq) + min(sq, (q + 1) * tok)) // 32) + SEGMENT for q in range(qtiles)) * hkv * batch
    share = max(MIN_SHARE, -(-units // cus))
    ns = cus // items
    dealt = None if ns and -(-tiles // ns) <= share + share // ALIGNED else unit * (share + SPARE) + DEAL_US

    def ordered(s):
        w = -(-wide_items * s // cus) * wide < -(-items * s // cus) * tile
        nq = -(-sq * g // 256) if w else qtiles
        launch = []
        for _ in range(hkv * batch):
            for split in range(s):
                for q in range(nq):
                    last = min((q + 1) * 256 - 1, sq * g - 1) // g + 1 if w else min(sq, (q + 1) * tok)
                    t = -(-(max(0, keys - sq) + last) // 32)
                    per = -(-t // s)
                    launch.append(max(0, min(per, t - split * per)) * (wide if w else tile) + pth_dec.PREFILL_US_PER_WORKGROUP)
        if len(launch) > 64 * cus:
            return 0.0
        span = at = 0
        for xcd in range(8):
            free = [0.0] * (cus // 8)
            n = len(launch) // 8 + (xcd < len(launch) % 8)
            for us in launch[at:at + n]:
                span = max(span, us + free[0])
                heapq.heapreplace(free, us + free[0])
            at += n
        merge = pth_dec.PREFILL_US_MERGE_LAUNCH + pth_dec.PREFILL_US_PER_PARTIAL_MB * rows * s * 1032 / 1e6 if s > 1 else 0.0
        return span + merge
    return out, dealt, ordered


@pytest.mark.parametrize("exact", [False, True], ids=["default", "exact"])
@pytest.mark.parametrize("seed", range(4))
def test_chunk_plan_equals_its_model(seed, exact):
    r, seen = random.Random(seed), set()
    for _ in range(120):
        hkv = r.choice([1, 2, 4, 8])
        batch, hq, sq = r.choice([1, 1, 3]), hkv * r.choice([1, 4, 6, 8]), r.choice([r.randint(1, 100), r.randint(1, 6000), 2048])
        keys, bs = sq + r.choice([0, r.randint(1, 2000), r.randint(1, 300000)]), r.choice([1, 8, 16, 48, 1584])
        counts, dealt, ordered = chunk_model(batch, sq, hq, hkv, keys, bs, exact)
        best = min(t for t, _ in counts.values())
        got = pth_dec._prefill_plan(batch, sq, hq, hkv, keys, bs, sq, exact)
        first = min(s for s, (t, _) in counts.items() if t == min(t for t, _ in counts.values()))
        deal = dealt is not None and dealt < MARGIN * best and dealt < MARGIN * ordered(first)
        assert (got == 0) == deal, (counts, dealt, got)
        if got:
            assert counts[got][0] == pytest.approx(best, rel=1e-12)
        seen.add(0 if got == 0 else counts[got][1])
    assert seen == {0, 192, 256}  # every kernel is planned somewhere


# batch, tokens, cached keys (24 q / 4 kv heads), exact, us unsplit, us dealt
FRESH_BATCHES = [(3, 1000, 0, False, 109.3, 133.0), (2, 1900, 0, False, 169.4, 201.7), (4, 1600, 0, False, 236.4, 280.9),
                 (2, 2000, 1000, False, 282.1, 320.1), (2, 3000, 0, False, 340.1, 372.5), (3, 1000, 0, True, 127.2, 145.8),
                 (1, 4000, 0, False, 371, 303), (1, 3000, 0, True, 337, 228), (1, 6000, 0, False, 776, 593)]


@pytest.mark.parametrize("batch,sq,ctx,exact,unsplit,dealt", FRESH_BATCHES)
def test_fresh_batches_are_planned_as_measured(batch, sq, ctx, exact, unsplit, dealt):
    got = pth_dec._prefill_plan(batch, sq, 24, 4, ctx + sq, 16, sq, exact)
    assert (got == 0) == (dealt < unsplit)


def test_plan_and_launch_share_the_tile_times():
    assert TIMES[False][0] == pth_dec.PREFILL_US_PER_TILE
    csrc = os.path.join(os.path.dirname(pth_dec.__file__), "csrc")
    assert "fa_wide_saves(wide_rounds, rounds, exact)" in open(os.path.join(csrc, "pd_prefill.hip")).read()
    # an exact call is rated with its own times: here a 256-row count that saves a round by the default's ratio only
    tile, wide, _ = TIMES[True]
    assert wide / tile > TIMES[False][1] / TIMES[False][0]


def test_errors_become_python_exceptions():
    c = kvcache.allocate_cache(2, 16, 2)
    views = (c.key_cache, c.value_cache, c.k_scale, c.v_scale)
    slots = torch.zeros(3, dtype=torch.int64)
    entry, write = pth_dec._entry("pth_cache_write"), pth_dec.native().cache_write
    x = torch.zeros((3, 2, 256), dtype=torch.float16)
    with pytest.raises(RuntimeError, match="must be fp16, bf16 or fp32 of the same dtype"):
        write(entry, x, x.float(), *views, slots)  # the entry's own check and message
    with pytest.raises(RuntimeError, match="tensor rank 5 exceeds 4"):
        write(entry, x.view(3, 1, 1, 2, 256), x, *views, slots)
    with pytest.raises(TypeError, match="expected a tensor, got list"):
        write(entry, [0.0], x, *views, slots)
    with pytest.raises(TypeError, match="expected 8 arguments"):
        write(entry, x)
    with pytest.raises(ValueError, match="null entry point"):
        write(0, x, x, *views, slots)
    with pytest.raises((RuntimeError, NotImplementedError)):  # no storage: torch's own error, not an abort
        write(entry, x.to_sparse(), x, *views, slots)
