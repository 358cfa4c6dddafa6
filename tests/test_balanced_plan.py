"""The deals of pd_balanced_kernel and pd_prefill_balanced_kernel restated on the CPU (constants read from the sources).

Decode: for any batch, workgroup count and segment cap, every tile of every (sequence, kv head) goes to exactly one
workgroup, the segments of an item are numbered from 0 in the order of its tiles, and there are at most `cap` of them.
Prefill: for any query tiles, kv heads and workgroup count, every key tile of every (kv head, query tile) goes to exactly
one workgroup, an item in one piece is stored by it, and the pieces of the others lie in the workspace slots where the
merge, which works them out anew, looks for them.
tests/test_balanced_decode_gpu.py and tests/test_balanced_prefill_gpu.py compare the kernels with the oracle.
"""
import os
import random
import re

import pytest

from mi50_vllm_lab_amd import pth_dec

SRC = open(os.path.join(os.path.dirname(pth_dec.__file__), "csrc", "pd_decode.hip")).read()
COST, SNAP = (int(re.search(r"constexpr unsigned %s = (\d+);" % n, SRC).group(1)) for n in ("kSegmentUnits", "kSnapTiles"))


def deal(tiles, hkv, nwg, cap):
    """{(sequence, kv head): [(segment, first tile, past the last)]}"""
    def units(t):
        return t + COST if t else 0

    total, longest, items = hkv * sum(map(units, tiles)), max(tiles), len(tiles) * hkv
    share = max(-(-total // nwg), (longest + cap - 2) // (cap - 1), 2)
    ns = min(nwg // items, cap)
    aligned = ns >= 1 and -(-longest // ns) <= share
    snap = min(SNAP, share // 8)
    lead = COST + snap
    starts = [hkv * sum(map(units, tiles[:b])) for b in range(len(tiles))]

    def locate(pos):
        k = sum(starts[i] + hkv * units(t) <= pos for i, t in enumerate(tiles))
        return k, starts[k], tiles[k]

    def bound(x):
        raw = min(x * share, total)
        if raw in (0, total):
            return raw
        _, start, t = locate(raw)
        off = (raw - start) % units(t)
        if off <= lead:
            return raw - off
        return raw + units(t) - off if units(t) - off <= snap else raw

    out = {}
    for wg in range(nwg):
        if aligned:
            item, seg = divmod(wg, ns)
            if item < items and tiles[item // hkv]:
                n = tiles[item // hkv]
                per = -(-n // ns)
                if seg * per < n:
                    out.setdefault((item // hkv, item % hkv), []).append((seg, seg * per, min(n, seg * per + per)))
            continue
        pos, end = bound(wg), bound(wg + 1)
        while pos < end:
            b, start, t = locate(pos)
            g = (pos - start) // units(t)
            item = start + g * units(t)
            first = 0 if pos - item <= lead else pos - item - COST
            last = t if end - item >= units(t) else end - item - COST
            seg = wg - min(item + lead, item + units(t) - 1) // share
            out.setdefault((b, g), []).append((seg, first, last))
            if last < t:
                break
            pos = item + units(t)
    return out


@pytest.mark.parametrize("seed", range(8))
def test_every_tile_once_and_segments_in_order(seed):
    r = random.Random(seed)
    for _ in range(150):
        n, hkv = r.randint(2, r.choice([4, 20, 130])), r.choice([1, 2, 3, 4, 8])
        nwg, cap, most = r.choice([1, 7, 64, 256, 304]), r.choice([2, 3, 5, 16, 64, 128]), r.choice([3, 40, 600, 6000])
        tiles = [r.choice([0, 1, r.randint(1, most), r.randint(1, most), most]) for _ in range(n)]
        if not any(tiles):
            continue
        out = deal(tiles, hkv, nwg, cap)
        assert sorted(out) == [(b, g) for b in range(n) if tiles[b] for g in range(hkv)]
        for (b, _), pieces in out.items():
            pieces.sort()
            assert [s for s, _, _ in pieces] == list(range(len(pieces))) and len(pieces) <= cap
            assert [f for _, f, _ in pieces] == [0] + [x for _, _, x in pieces[:-1]] and pieces[-1][2] == tiles[b]
            assert all(f < x for _, f, x in pieces)


CSRC = os.path.join(os.path.dirname(pth_dec.__file__), "csrc")
FA_COST, FA_MIN_SHARE, FA_ALIGNED, FA_PIECES = (
    int(re.search(r"constexpr unsigned %s = (\d+);" % n, open(os.path.join(CSRC, f)).read()).group(1))
    for n, f in (("kFaSegmentUnits", "pd_plan.hpp"), ("kFaMinShare", "pd_plan.hpp"), ("kFaAlignedPart", "pd_plan.hpp"),
                 ("kFaMaxPieces", "pd_prefill.hip")))


class PrefillLine:
    """fa_line, fa_locate and fa_bound for query tiles that see tiles[c] key tiles."""

    def __init__(self, tiles, hkv, nwg):
        self.tiles, self.hkv, self.nwg, self.items = tiles, hkv, nwg, len(tiles) * hkv
        self.starts = [sum(t + FA_COST for t in tiles[:c]) for c in range(len(tiles) + 1)]
        self.per_head = self.starts[-1]
        self.total, longest = self.per_head * hkv, max(tiles)
        self.share = max(-(-self.total // nwg), (longest + FA_COST + FA_PIECES - 3) // (FA_PIECES - 2), FA_MIN_SHARE)
        self.ns = min(nwg // self.items, FA_PIECES, max(1, longest // 8))
        self.aligned = nwg >= self.items and -(-longest // self.ns) <= self.share + self.share // FA_ALIGNED
        self.snap = min(8, self.share // 8)
        self.lead = FA_COST + self.snap

    def locate(self, pos):
        c = sum(x <= pos for x in self.starts[1:])
        return c, self.starts[c], self.tiles[c]

    def bound(self, x):
        raw = min(x * self.share, self.total)
        if raw in (0, self.total):
            return raw
        _, start, t = self.locate(raw % self.per_head)
        off, units = raw % self.per_head - start, t + FA_COST
        if off <= self.lead:
            return raw - off
        return raw + units - off if units - off <= self.snap else raw


def prefill_deal(n):
    """{(kv head, query tile): [(first tile, past the last, slot or -1)]} as pd_prefill_balanced_kernel's workgroups take them"""
    out = {}
    for wg in range(n.nwg):
        if n.aligned:
            item, piece = divmod(wg, n.ns)
            if item >= n.items:
                continue
            t = n.tiles[item % len(n.tiles)]
            per = -(-t // n.ns)
            first, last = piece * per, min(t, piece * per + per)
            if piece == 0 or first < last:
                whole = first == 0 and last == t
                out.setdefault(divmod(item, len(n.tiles)), []).append((first, last, -1 if whole else 2 * wg))
            continue
        pos, end, segment = n.bound(wg), n.bound(wg + 1), 0
        while pos < end:
            g, in_head = divmod(pos, n.per_head)
            c, start, t = n.locate(in_head)
            start += g * n.per_head
            first = 0 if pos - start <= n.lead else pos - start - FA_COST
            last = t if end - start >= t + FA_COST else end - start - FA_COST
            whole = first == 0 and last == t
            out.setdefault((g, c), []).append((first, last, -1 if whole else 2 * wg + (segment > 0)))
            if last < t:
                break
            pos, segment = start + t + FA_COST, segment + 1
    return out


def merge_slots(n, g, c):
    """The slots that pd_prefill_merge_kernel reads for an item; none for an item in one piece."""
    t = n.tiles[c]
    if n.aligned:
        per = max(1, -(-t // n.ns))
        pieces = -(-t // per)
        return [2 * ((g * len(n.tiles) + c) * n.ns + i) for i in range(pieces)] if pieces > 1 else []
    start, units = n.starts[c] + g * n.per_head, t + FA_COST
    j0 = min(start + n.lead, start + units - 1) // n.share
    inside = (start + units - n.snap + n.share - 1) // n.share - 1 if units > n.snap else j0
    if inside <= j0:
        return []
    return [2 * (j0 + i) + (1 if i == 0 and n.bound(j0) != start else 0) for i in range(inside - j0 + 1)]


@pytest.mark.parametrize("seed", range(8))
def test_prefill_every_tile_once_and_pieces_where_the_merge_looks(seed):
    r = random.Random(seed)
    for _ in range(150):
        nq, hkv = r.randint(1, r.choice([4, 20, 130])), r.choice([1, 2, 3, 4, 8])
        nwg, most = r.choice([1, 7, 64, 256, 304]), r.choice([3, 40, 600, 4000])
        tiles = [r.choice([0, 1, r.randint(0, most), r.randint(0, most), most]) for _ in range(nq)]
        if r.random() < 0.3:
            tiles = sorted(tiles) if r.random() < 0.5 else [most] * nq
        n = PrefillLine(tiles, hkv, nwg)
        out, used = prefill_deal(n), set()
        assert sorted(out) == [(g, c) for g in range(hkv) for c in range(nq)]  # tiles without keys too: their rows are 0
        for (g, c), pieces in out.items():
            pieces.sort()
            assert [f for f, _, _ in pieces] == [0] + [x for _, x, _ in pieces[:-1]] and pieces[-1][1] == tiles[c]
            assert len(pieces) <= FA_PIECES and (len(pieces) == 1 or all(f < x for f, x, _ in pieces))
            slots = [s for _, _, s in pieces]
            assert merge_slots(n, g, c) == ([] if len(pieces) == 1 else slots)
            assert (slots == [-1]) == (len(pieces) == 1) and all(s < 2 * nwg for s in slots)
            assert not used & set(slots) - {-1}
            used |= set(slots)


@pytest.mark.parametrize("nwg", [1, 7, 8, 9, 100, 256, 304])
def test_prefill_workgroups_in_xcd_order_are_each_there_once(nwg):
    order = [b % 8 * (nwg // 8) + min(b % 8, nwg % 8) + b // 8 for b in range(nwg)]
    assert sorted(order) == list(range(nwg))
