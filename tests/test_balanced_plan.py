"""The deal of pd_balanced_kernel restated on the CPU (constants read from the kernel source): for any batch,
workgroup count and segment cap, every tile of every (sequence, kv head) goes to exactly one workgroup, the
segments of an item are numbered from 0 in the order of its tiles, and there are at most `cap` of them.
tests/test_balanced_decode_gpu.py compares the kernel itself with the oracle and the general path.
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
