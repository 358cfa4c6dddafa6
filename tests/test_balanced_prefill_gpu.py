"""GPU parity of the balanced prefill (pd_prefill_balanced_kernel and its merge) and of the rows form against
the float64 oracle: query tiles with few, equal and very different key counts, so that the deal takes both of
its splits, pieces at the edges of items, items without keys, and launches of one workgroup up to all of
them; several sequences per launch, empty ones among them; both numerics; every page-table path.
"""
import numpy as np
import pytest
import torch

import workload as kvc
from mi50_vllm_lab_amd import pth_dec
from oracle import attention as orc

pytestmark = pytest.mark.gpu

SLOT = 2 * 192 * 258  # workspace floats of one workgroup


def balanced(q, d, q_abs, out, starts, exact, floats=None, nsplit=0):
    """pth_fa_forward_balanced through the C entry, on a workspace of `floats` (default: what it asks for) of NaN."""
    import ctypes
    lib = pth_dec.load_library()
    c, rows = d.cache, starts is not None
    host = (ctypes.c_int * len(starts))(*starts) if rows else None
    keys = int(d.seq_lens.max())
    need = lib.pth_fa_balanced_workspace(len(starts) - 1 if rows else q.shape[0], host, 0 if rows else q.shape[2],
                                         q.shape[1], c.num_kv_heads, keys, d.block_table.shape[1] * c.block_size)
    assert need > 0 and need % SLOT == 0
    ws = torch.full((floats or need,), float("nan"), dtype=torch.float32, device="cuda")
    descs = [pth_dec.describe(t) for t in (q, c.key_cache, c.value_cache, d.block_table, d.seq_lens)]
    qa, od, wd = (pth_dec.describe(t) for t in (q_abs, out, ws))
    err = ctypes.create_string_buffer(256)
    rc = lib.pth_fa_forward_balanced(*[ctypes.byref(x) for x in descs], d.scale, ctypes.byref(qa), host,
                                     len(starts) - 1 if rows else 0, ctypes.byref(od), ctypes.byref(wd), keys, nsplit,
                                     1 if exact else 0, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), err, 256)
    assert rc == 0, err.value
    torch.cuda.synchronize()


BATCHES = {  # contexts, chunk, q_abs offsets from the context, (q, kv heads), block size
    "fresh": ([0], 700, [0], (24, 4), 16),
    "fresh_one_tile_more": ([0], 33, [0], (24, 4), 16),
    "long_context": ([5000], 70, [0], (24, 4), 16),
    "offsets": ([3000, 0, 517], 70, [0, -20, 183], (24, 4), 16),
    "no_visible_key": ([0, 0], 40, [-40, -300], (8, 2), 16),
    "group_of_7": ([100, 2000], 77, [0, 0], (28, 4), 16),
    "group_of_1_pages_of_8": ([900], 130, [0], (4, 4), 8),
    "reference_blocks": ([1584 * 2 - 5], 300, [0], (12, 2), 1584),
    "more_query_tiles_than_lanes": ([0], 2200, [0], (6, 1), 32),
}


@pytest.mark.parametrize("exact", [False, True], ids=["default", "exact"])
@pytest.mark.parametrize("wgs", [None, 1, 7, 100], ids=["all", "1", "7", "100"])
@pytest.mark.parametrize("name", list(BATCHES))
def test_batch_form(name, wgs, exact):
    ctxs, sq, off, (hq, hkv), bs = BATCHES[name]
    c = kvc.make_case(ctxs, [sq] * len(ctxs), num_q_heads=hq, num_kv_heads=hkv, block_size=bs, seed=len(name),
                      layout="NHD" if len(name) % 2 else "HND")
    q_abs = [x + o for x, o in zip(ctxs, off)]
    print(f"balanced prefill {name} wgs={wgs} exact={exact}", flush=True)
    d = c.to("cuda")
    q = kvc.prefill_query(d)
    out = torch.full((q.shape[0], sq, hq, 256), float("nan"), dtype=torch.float32, device="cuda")
    balanced(q, d, torch.tensor(q_abs, dtype=torch.int32, device="cuda"), out, None, exact, wgs and wgs * SLOT)
    rows = None if sq <= 300 else sorted({0, 31, 32, 33, sq - 1} | set(range(5, sq, 61)))
    ref, written = orc.paged_prefill(kvc.prefill_query(c), c.cache.key_cache, c.cache.value_cache, c.cache.k_scale,
                                     c.cache.v_scale, c.block_table, c.seq_lens, c.scale, torch.tensor(q_abs), rows)
    o = out.double().cpu().numpy()
    assert np.isfinite(o).all()
    if written.any():
        e = np.abs(o[written] - ref[written])
        print(f"  max-abs {e.max():.2e} mean-abs {e.mean():.2e}", flush=True)
        assert e.max() <= 2e-3 and e.mean() <= 2e-4
    if rows is None:
        assert (o[~written] == 0).all()  # rows that see no key


ROWS = {  # contexts, new tokens, (q, kv heads), block size
    "one": ([300], [100], (24, 4), 16),
    "mixed": ([300, 0, 4000, 17, 0], [70, 1, 200, 33, 500], (24, 4), 16),
    "empty_ones": ([50, 90, 10, 0], [0, 40, 0, 65], (24, 4), 16),
    "rank_reference_blocks": ([3000, 0], [64, 333], (12, 2), 1584),
    "pages_of_8": ([100, 700], [90, 31], (8, 8), 8),
    "thirty_two": ([13 * i for i in range(32)], [1 + 5 * (i % 9) for i in range(32)], (24, 4), 16),
}


@pytest.mark.parametrize("exact", [False, True], ids=["default", "exact"])
@pytest.mark.parametrize("nsplit", [0, 1, 3])
@pytest.mark.parametrize("name", list(ROWS))
def test_rows_form(name, nsplit, exact):
    """fp16 rows in and out, other rows around them; nsplit > 0 (one sequence): the split kernels on rows."""
    ctxs, news, (hq, hkv), bs = ROWS[name]
    if nsplit and len(ctxs) > 1:
        pytest.skip("splits take one sequence")
    c = kvc.make_case(ctxs, news, num_q_heads=hq, num_kv_heads=hkv, block_size=bs, seed=len(name) + 3, q_noncontig=True)
    print(f"rows {name} nsplit={nsplit} exact={exact}", flush=True)
    d = c.to("cuda")
    lead, total = 3, sum(news)
    q = torch.full((total + 5, hq + 4, 256), float("nan"), dtype=torch.float16, device="cuda")[:, 2:2 + hq]
    q[lead:lead + total] = d.q
    out = torch.full((total + 5, hq, 256), 7.0, dtype=torch.float16, device="cuda")
    starts = [lead + sum(news[:i]) for i in range(len(news) + 1)]
    floats = max(4, news[0] * hq * nsplit * 258) if nsplit else None
    balanced(q, d, d.seq_lens, out, starts, exact, floats, nsplit)
    o = out.double().cpu().numpy()
    assert (o[:lead] == 7).all() and (o[lead + total:] == 7).all()
    for i, n in enumerate(news):
        if n == 0:
            continue
        qi = c.q[starts[i] - lead:starts[i] - lead + n].transpose(0, 1).unsqueeze(0).float().contiguous()
        ref, written = orc.paged_prefill(qi, c.cache.key_cache, c.cache.value_cache, c.cache.k_scale, c.cache.v_scale,
                                         c.block_table[i:i + 1], c.seq_lens[i:i + 1], c.scale, torch.tensor([ctxs[i]]))
        assert written.all()
        emax, emean, over, over_mean = kvc.fp16_output_errors(o[starts[i]:starts[i + 1]], ref[0])
        assert over <= 0 and over_mean <= 2e-4, (i, emax, emean)


def test_rows_graph_replays():
    """Captured through the Python face and replayed, each replay equal to the eager call."""
    c = kvc.make_case([300, 0, 4000], [70, 1, 200], num_q_heads=24, num_kv_heads=4, block_size=16, seed=5).to("cuda")
    starts, k = [0, 70, 71, 271], c.cache
    want, out = torch.zeros_like(c.q), torch.zeros_like(c.q)

    def call(o):
        assert pth_dec.forward_rows(c.q, k.key_cache, k.value_cache, c.block_table, c.seq_lens, c.scale, starts, o, 4200)
    call(want)
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s), torch.cuda.graph(g, stream=s):
        call(out)
    torch.cuda.current_stream().wait_stream(s)
    for _ in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("wgs", [None, 10], ids=["all", "10"])
def test_error_does_not_grow_with_the_run(wgs):
    """Chunks over long prefixes, each workgroup on a run of hundreds of key tiles (10 workgroups: thousands, across
    items). The default numerics round the weights to fp16, and the output is fp16: each at most 2^-11 / sqrt(3) =
    2.8e-4 of the result's norm, 4e-4 together; nothing that grows with the keys may come on top."""
    ctxs, news = [60000, 30011, 45000, 52000], [200, 77, 130, 100]
    c = kvc.make_case(ctxs, news, num_q_heads=6, num_kv_heads=1, block_size=16, seed=11)
    d = c.to("cuda")
    out = torch.full_like(d.q, float("nan"))
    starts = [sum(news[:i]) for i in range(5)]
    balanced(d.q, d, d.seq_lens, out, starts, False, wgs and wgs * SLOT)
    o = out.double().cpu().numpy()
    assert np.isfinite(o).all()
    num = den = 0.0
    for i, n in enumerate(news):
        rows = [0, n // 2, n - 1]
        qi = c.q[starts[i]:starts[i + 1]].transpose(0, 1).unsqueeze(0).float().contiguous()
        ref, _ = orc.paged_prefill(qi, c.cache.key_cache, c.cache.value_cache, c.cache.k_scale, c.cache.v_scale,
                                   c.block_table[i:i + 1], c.seq_lens[i:i + 1], c.scale, torch.tensor([ctxs[i]]), rows)
        e = o[starts[i]:starts[i + 1]][rows] - ref[0][rows]
        num, den = num + (e ** 2).sum(), den + (ref[0][rows] ** 2).sum()
    print(f"  wgs={wgs} error {np.sqrt(num / den):.2e} of the result", flush=True)
    assert np.sqrt(num / den) <= 4e-4


def test_rows_calls_that_the_loop_takes():
    """Calls that one forward_pth per sequence takes are taken as well, or left to it (False): out with more or
    fewer rows than query, strided lengths, an output on the host."""
    c = kvc.make_case([300, 0], [70, 65], num_q_heads=24, num_kv_heads=4, block_size=16, seed=6).to("cuda")
    k, starts = c.cache, [0, 70, 135]

    def call(q, out, lens=c.seq_lens):
        return pth_dec.forward_rows(q, k.key_cache, k.value_cache, c.block_table, lens, c.scale, starts, out, 370)
    want = torch.zeros_like(c.q)
    assert call(c.q, want)
    longer = torch.full((150, 24, 256), 7.0, dtype=torch.float16, device="cuda")
    assert call(c.q, longer) and torch.equal(longer[:135], want) and (longer[135:] == 7).all()
    shorter = torch.zeros_like(want)
    assert call(torch.cat([c.q, c.q[:9]]), shorter) and torch.equal(shorter, want)
    untouched = torch.full_like(want, 7.0)
    lens = torch.stack([c.seq_lens, c.seq_lens], 1)[:, 0]
    assert not lens.is_contiguous() and not call(c.q, untouched, lens) and (untouched == 7).all()
    assert not call(c.q, torch.empty(want.shape, dtype=torch.float16))
    with pytest.raises(RuntimeError, match="within the rows of q and out"):
        call(c.q, untouched[:134])


def test_planned_calls_without_memory_for_their_workspace():
    """With no room for the partials a planned call runs unsplit, several chunks are left to the loop, and a split
    count that the caller asked for raises torch's error. The room is limited in torch's allocator."""
    c = kvc.make_case([3000], [1501], num_q_heads=24, num_kv_heads=4, block_size=16, seed=8).to("cuda")
    k, q, starts = c.cache, kvc.prefill_query(c), [0, 1501]
    q_abs = torch.tensor([3000], dtype=torch.int32, device="cuda")
    out, rows = torch.empty((1, 1501, 24, 256), device="cuda"), torch.empty_like(c.q)

    def batch(nsplit, max_keys):
        pth_dec.forward_pth(q, k.key_cache, k.value_cache, c.block_table, c.seq_lens, c.scale, q_abs, out=out,
                            nsplit=nsplit, max_keys=max_keys)
        return out.clone()

    def chunk(starts, max_keys):
        rows.fill_(7)
        return pth_dec.forward_rows(c.q, k.key_cache, k.value_cache, c.block_table.expand(len(starts) - 1, -1),
                                    c.seq_lens.expand(len(starts) - 1).contiguous(), c.scale, starts, rows, max_keys)
    unsplit, plans = batch(1, 4501), [pth_dec._prefill_plan(1, 1501, 24, 4, m, 16, 1501) for m in (4501, 200000)]
    assert plans[0] == 0 and plans[1] > 1  # dealt, and split
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room = torch.cuda.memory_reserved() + (64 << 20)
    torch.cuda.set_per_process_memory_fraction(room / torch.cuda.get_device_properties(0).total_memory)
    try:
        for max_keys in (4501, 200000):
            assert torch.equal(batch(None, max_keys), unsplit)
            assert chunk(starts, max_keys)
            assert (rows.cpu().float() - unsplit[0].cpu()).abs().max() <= 2e-3
        assert not chunk([0, 300, 1501], 4501) and (rows.cpu() == 7).all()
        with pytest.raises(torch.OutOfMemoryError):
            batch(8, 4501)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert chunk([0, 300, 1501], 4501)
