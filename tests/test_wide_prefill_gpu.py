"""GPU parity of the 256-row prefill kernel (pd_prefill_wide_kernel), which launches of several rounds of
workgroups take, against the float64 oracle on sampled rows: tokens that straddle its workgroups (256 is no
multiple of the group), a part-filled last workgroup, waves without rows, an odd number of key tiles per step
pair, both numerics, every page-table path, fp32 and fp16 rows, split and unsplit.
"""
import numpy as np
import pytest
import torch

import workload as kvc
from mi50_vllm_lab_amd import pth_dec
from oracle import attention as orc

pytestmark = pytest.mark.gpu

# contexts, chunk, (q, kv heads), block size, splits: each takes the 256-row kernel (see rounds() below)
CASES = {
    "three_rounds_for_four": ([300], 2048, (24, 4), 16, 4),
    "odd_tiles_part_filled": ([1000], 2031, (24, 4), 16, 4),
    "unsplit": ([40, 0], 4090, (24, 4), 16, 1),
    "group_of_7": ([90], 2050, (28, 4), 16, 4),
    "pages_of_8": ([70], 2048, (24, 4), 8, 4),
    "pages_of_48_nhd": ([500], 2047, (24, 4), 48, 4),
    "reference_blocks": ([3000], 2048, (12, 2), 1584, 8),
    "positions_before_the_first_key": ([0], 2040, (24, 4), 16, 4),
}


def rounds(rows, unit, heads_kv, batch, nsplit, tok=None):
    wgs = -(-rows // unit) if tok is None else -(-rows // tok)
    return -(-wgs * heads_kv * batch * nsplit // 256)


@pytest.mark.parametrize("exact", [False, True], ids=["default", "exact"])
@pytest.mark.parametrize("form", ["fp32", "rows"])
@pytest.mark.parametrize("name", list(CASES))
def test_against_the_oracle(name, form, exact):
    ctxs, sq, (hq, hkv), bs, nsplit = CASES[name]
    g = hq // hkv
    # the rule of launch_prefill
    assert rounds(sq * g, 256, hkv, len(ctxs), nsplit) * (2.2 / 1.9 if exact else 1.85 / 1.62) < \
        rounds(sq, None, hkv, len(ctxs), nsplit, 192 // g), "this case does not take the kernel"
    if form == "rows" and len(ctxs) > 1:
        pytest.skip("splits of rows take one sequence")
    c = kvc.make_case(ctxs, [sq] * len(ctxs), num_q_heads=hq, num_kv_heads=hkv, block_size=bs, seed=len(name) + sq,
                      layout="NHD" if "nhd" in name else "HND", outlier_frac=0.0 if not exact else 0.01)
    off = -35 if name.startswith("positions") and form == "fp32" else 0
    q_abs = [x + off for x in ctxs]
    print(f"wide prefill {name} {form} exact={exact}", flush=True)
    d = c.to("cuda")
    k = d.cache
    if form == "fp32":
        out = torch.full((len(ctxs), sq, hq, 256), float("nan"), dtype=torch.float32, device="cuda")
        pth_dec.forward_pth(kvc.prefill_query(d), k.key_cache, k.value_cache, d.block_table, d.seq_lens, d.scale,
                            torch.tensor(q_abs, dtype=torch.int32, device="cuda"), out=out, exact=exact, nsplit=nsplit)
    else:
        out = torch.full((sq, hq, 256), float("nan"), dtype=torch.float16, device="cuda")
        assert pth_dec.native().prefill_balanced(
            pth_dec._entry("pth_fa_forward_balanced"), pth_dec._entry("pth_fa_balanced_workspace"), d.q, k.key_cache,
            k.value_cache, d.block_table, d.seq_lens, d.scale, None, out, [0, sq], max(ctxs) + sq, nsplit, int(exact))
        out = out.unsqueeze(0)
    torch.cuda.synchronize()
    o = out.double().cpu().numpy()
    assert np.isfinite(o).all()
    # the rows at the workgroups' edges and a few others
    edges = {t for w in range(0, sq * g, 256) for t in ((w - 1) // g, w // g)}
    rows = sorted({0, 31, 34, 35, sq - 1} | {t for t in sorted(edges) if 0 <= t < sq} - set(range(200, sq - 60)) | set(range(7, sq, 211)))
    ref, written = orc.paged_prefill(kvc.prefill_query(c), c.cache.key_cache, c.cache.value_cache, c.cache.k_scale,
                                     c.cache.v_scale, c.block_table, c.seq_lens, c.scale, torch.tensor(q_abs), rows)
    e = np.abs(o[written] - ref[written])
    half = kvc.fp16_half_ulp(ref[written]) if form == "rows" else 0.0
    print(f"  max-abs {e.max():.2e} mean-abs {e.mean():.2e}", flush=True)
    assert (e <= 2e-3 + half).all() and np.maximum(e - half, 0).mean() <= 2e-4
    if off:
        assert (o[:, :-off] == 0).all()  # rows that see no key
