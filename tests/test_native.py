"""pd_native (csrc/pd_python.cpp) on the CPU: the split plans equal their models, and errors come back as the
Python exceptions that the operators document. The calls themselves are covered by every GPU test.
"""
import math
import random

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
