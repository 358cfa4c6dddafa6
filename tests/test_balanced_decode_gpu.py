"""GPU parity of the batch decode (pd_balanced_kernel: the tiles of all sequences dealt evenly over the
workgroups by the lengths on the device) against the float64 oracle and against the general path, the
split-per-sequence launches pth_dec_launch_partial and pth_dec_launch_combine.

The batches are those at whose edges the deal can go wrong: sequences of one key, of exactly one
tile and of one key more, empty ones, one long sequence among short ones (its segments at the cap of the
partial buffers), equal lengths (cut evenly, one workgroup each), more sequences than a wave's lanes, more
items than workgroups. Each is launched at a split count that the operator deals, which the test sees in the segments
written. Every partial buffer starts as NaN: a segment that nobody wrote must not be read.
"""
import numpy as np
import pytest
import torch

import workload as kvc
from mi50_vllm_lab_amd import pth_dec
from oracle import attention as orc

pytestmark = pytest.mark.gpu

MIXED = [1, 31, 32, 33, 700, 5000, 97, 12000]
BATCHES = {
    # name: contexts, query tokens, (q heads, kv heads), block size, segments, splits (x kv heads x sequences above 256), window
    "mixed": (MIXED, [1] * 8, (24, 4), 16, 64, 16, -1),
    "mixed_mtp_two_row_blocks": (MIXED, [4, 0, 1, 2, 4, 3, 0, 4], (24, 4), 16, 64, 16, -1),
    "long_among_short_at_three_segments": ([40000, 10, 900, 64] + [9] * 130, [1] * 134, (12, 2), 16, 3, 2, -1),
    "long_among_short_at_five_segments": ([30000, 10, 900, 64] + [40] * 13, [2, 1, 2, 1] + [1] * 13, (24, 4), 32, 5, 4, -1),
    "more_segments_than_lanes": ([60000, 10, 300], [1, 1, 1], (6, 1), 16, 128, 100, -1),
    "equal": ([2048] * 6, [1] * 6, (24, 4), 16, 64, 16, -1),
    "equal_reference_blocks": ([3000] * 3, [4] * 3, (12, 2), 1584, 64, 48, -1),
    "nearly_equal_many_items": ([500 + 3 * (i % 7) for i in range(70)], [1] * 70, (32, 8), 16, 64, 4, -1),
    "lanes_plus_one": ([(i * 37) % 400 for i in range(65)], [1 + i % 2 for i in range(65)], (8, 2), 16, 64, 4, -1),
    "more_than_two_waves_of_sequences": ([(i * 53) % 230 + 1 for i in range(130)], [1] * 130, (8, 2), 16, 16, 4, -1),
    "no_query_tokens_but_one": ([500, 900, 40], [0, 3, 0], (24, 4), 16, 64, 32, -1),
    "pages_not_of_16": (MIXED, [1] * 8, (24, 4), 8, 64, 16, -1),
    "pages_of_one": ([1, 31, 33, 2000, 97] + [20 + i for i in range(15)], [2] * 20, (24, 4), 1, 7, 5, -1),
    "window": (MIXED, [1, 2, 1, 2, 1, 2, 1, 2], (24, 4), 16, 64, 16, 512),
    "window_past_the_sliced_size": ([9000, 100, 20000, 31], [4] * 4, (24, 4), 16, 64, 32, 8192),
}


def decode(c, nseg, nsplit):
    d = c.to("cuda")
    hq = c.num_q_heads
    out = torch.full((c.num_tokens, hq, 256), float("nan"), dtype=torch.float16, device="cuda")
    parts = [torch.full_like(t, float("nan")) for t in kvc.partial_buffers(c.num_tokens, hq, nseg, "cuda")]
    pth_dec.decode(d.q, d.cache.key_cache, d.cache.value_cache, d.cache.k_scale, d.cache.v_scale, d.block_table,
                   d.seq_lens, d.query_start_loc, out, d.scale, *parts, d.num_seqs, d.qmax, nsplit, d.window, d.causal)
    torch.cuda.synchronize()
    return d, out, parts


def dealt(parts, nsplit):
    """Whether the call ran pd_balanced_kernel: only that writes more than nsplit segments of the partial buffers."""
    return not parts[1][:, :, nsplit:].isnan().all().item()


def general_path(d, nseg, nsplit):
    hq, c = d.num_q_heads, d.cache
    out = torch.full((d.num_tokens, hq, 256), float("nan"), dtype=torch.float16, device="cuda")
    parts = kvc.partial_buffers(d.num_tokens, hq, nseg, "cuda")
    assert pth_dec.launch_partial(d.q, c.key_cache, d.block_table, d.seq_lens, d.query_start_loc, *parts,
                                  num_seqs=d.num_seqs, heads_q=hq, heads_kv=c.num_kv_heads, block_size=c.block_size,
                                  scale=d.scale, qmax=d.qmax, nsplit=nsplit, window=d.window, causal=d.causal) == 0
    assert pth_dec.launch_combine(d.seq_lens, d.query_start_loc, *parts, out, num_seqs=d.num_seqs, qmax=d.qmax,
                                  nsplit=nsplit) == 0
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("causal", [True, False], ids=["causal", "all_keys"])
@pytest.mark.parametrize("name", list(BATCHES))
def test_batches(name, causal):
    ctxs, qlens, (hq, hkv), bs, nseg, nsplit, window = BATCHES[name]
    c = kvc.make_case(ctxs, qlens, num_q_heads=hq, num_kv_heads=hkv, block_size=bs, seed=len(name), window=window,
                      causal=causal, layout="NHD" if len(name) % 2 else "HND", outlier_frac=0.01)
    ref, written = orc.paged_decode(c.q, c.cache.key_cache, c.cache.value_cache, c.cache.k_scale, c.cache.v_scale,
                                    c.block_table, c.seq_lens, c.query_start_loc, c.num_seqs, c.scale, c.window, c.causal)
    print(f"balanced {name} causal={causal}", flush=True)
    d, out, parts = decode(c, nseg, nsplit)
    assert dealt(parts, nsplit), "this batch does not run the kernel"
    o = out.double().cpu().numpy()
    emax, emean, over, over_mean = kvc.fp16_output_errors(o[written], ref[written])
    print(f"  max-abs {emax:.2e} mean-abs {emean:.2e}", flush=True)
    assert np.isfinite(o[written]).all() and over <= 0 and over_mean <= 2e-4, (emax, emean)
    # the general path differs by the order of the fp32 sums only: at most one fp16 step per value
    g = general_path(d, nseg, nsplit).double().cpu().numpy()[written]
    step = 2 * kvc.fp16_half_ulp(np.maximum(np.abs(g), np.abs(o[written]))) + 1e-6 * np.abs(ref[written]).max()
    assert (np.abs(g - o[written]) <= step).all()
    # and again on the same buffers, now full of the first call's partials
    again = torch.zeros_like(out)
    pth_dec.decode(d.q, d.cache.key_cache, d.cache.value_cache, d.cache.k_scale, d.cache.v_scale, d.block_table,
                   d.seq_lens, d.query_start_loc, again, d.scale, *parts, d.num_seqs, d.qmax, nsplit, d.window, d.causal)
    torch.cuda.synchronize()
    sel = torch.from_numpy(written).cuda()
    assert torch.equal(again[sel], out[sel])


# segments, splits, whether the batch (65 sequences x 4 kv heads: past one round at any count) is dealt
ROUTES = [(3, 2, True), (5, 4, True), (9, 8, False), (10, 8, True), (13, 12, False), (14, 12, True), (16, 15, False), (17, 16, True),
          (100, 4, True), (64, 1, False), (64, 2, True)]


@pytest.mark.parametrize("nseg,nsplit,deal", ROUTES)
def test_few_segments_stay_with_the_splits(nseg, nsplit, deal):
    """One long sequence among short ones is cut by the deal into at most one share less than there are segments: with
    no segments to spare for that the launch keeps its splits. So does one split, past one round, of sequences whose
    lengths only the caller knows."""
    c = kvc.make_case([2000] + [5] * 64, [1] * 65, num_q_heads=24, num_kv_heads=4, block_size=16, seed=nseg)
    d, out, parts = decode(c, nseg, nsplit)
    assert dealt(parts, nsplit) == deal
    ref, written = orc.paged_decode(c.q, c.cache.key_cache, c.cache.value_cache, c.cache.k_scale, c.cache.v_scale,
                                    c.block_table, c.seq_lens, c.query_start_loc, c.num_seqs, c.scale, c.window, c.causal)
    emax, emean, over, over_mean = kvc.fp16_output_errors(out.double().cpu().numpy()[written], ref[written])
    assert over <= 0 and over_mean <= 2e-4, (emax, emean)
    # either way every segment of the launch is written, the empty ones with m = -inf and l = 0
    m, l = (t[:, :, :min(nseg, 128) if deal else nsplit] for t in parts[1:])
    assert not m.isnan().any() and not l.isnan().any()
    assert (nsplit == 1 or (m == float("-inf")).any()) and (l[m == float("-inf")] == 0).all() and (l[m > float("-inf")] > 0).all()
