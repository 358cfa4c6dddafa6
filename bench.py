#!/usr/bin/env python3
"""Benchmark of the int8-KV paged attention operators on one MI355X.

Headline (`value`): MTP verify decode, 1 sequence x 4 causal query tokens, 24 q heads / 4 kv
heads (GQA 6 -> 24 rows per kv head), head_dim 256, ctx 61,440 + 4, int8 per-token-head cache
(K/V ~ N(0,1) quantised absmax/127), block_size 16, random page permutation, fp16 out. One step =
one operator call (one attention layer: both kernels, all 24 heads). Exactly `--steps` calls are
captured in one HIP graph (each call reads the next of `--rotate` identical caches, so every layer
reads its KV from HBM and not from the 256 MB Infinity Cache) and replayed once between device
synchronisations, timed with HIP events on the stream the kernels run on; `--warmup` calls are
replayed before, from a graph of their own.

`roofline`: the split-K partial kernel alone (the kernel that moves the KV bytes), a graph of a
fixed 2,000 launches over the rotating caches, timed the same way: algorithmic bytes per launch
/ average launch time against 8 TB/s. `traffic` and the MFMA counters come from the rocprofv3
summaries committed under profiles/ for the same workload.

`configs`: the other workloads, each with its own fixed repetition count:
  1  single-token decode, 1 x 1 token, ctx 4,096 (6 rows per kv head)
  3  DFlash2 drafter, 4 sequences (ctx 2,048 / 9,216 / 33,792 / 122,880) x 8 non-causal rows,
     2,048-key sliding window, pages outside every window freed (NaN)
  4  long context, 1 x 4 tokens, ctx 200,000, 1 % of the (token, kv head) rows x 50 before
     quantisation: one call captured in a HIP graph and the graph replayed 1,000 times
  5  chunked prefill, a 2,048-token causal chunk over 61,440 cached tokens (63,488 keys), through
     pth_fa_forward and (under `exact`) pth_fa_forward_exact; `chunk64` is a 64-token chunk over
     the same cache (keys split over 32 workgroups per query tile), `chunk2560` a 2,560-token one (4 splits)
  w  the KV-cache writer (pth_cache_write) on 4, 2,048 and 32,768 new tokens (fp16 K/V as
     strided views of a fused QKV buffer): µs per call, algorithmic GB/s, fraction of 8 TB/s
Decode configs report µs per layer, algorithmic GB/s and the fraction of 8 TB/s; the prefill
reports ms per chunk and TFLOP/s against the 2.5 PFLOP/s dense fp16 MFMA peak. The split count
of each decode config is the one the vLLM shim picks (vllm_shim.decode_splits with the host-side
lengths); config 2 uses the reference's 64.

CPU baselines: the float64 oracle (numpy + BLAS on every host core) on the same layer for
configs 1, 2 and 4 (median of 5 runs after one warm-up), and on a sample of query rows for
config 5.

Prints one JSON line.
"""
import argparse
import json
import math
import os
import platform
import subprocess
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
PKG_DIR = os.path.join(ROOT, "mi50-vllm-lab_amd")
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.join(ROOT, "tests"))

METRIC = "µs/layer + achieved KV GB/s (% of HBM peak), MTP 24-row decode at 61k ctx"
HBM_PEAK_GBS = 8000.0
MFMA_FP16_PEAK_TFLOPS = 2500.0
NSEG = 128
ROOF_LAUNCHES = 2000
CALIB_BYTES = 256 << 20
CALIB_COPIES = 8
PROFILES = os.path.join(ROOT, "profiles")


def _pmc_dispatches(run_dir, counter):
    """{dispatch id: (kernel name, summed counter value)} from a rocprofv3 --pmc csv run directory."""
    import csv
    import glob

    files = glob.glob(os.path.join(run_dir, "**", "*counter_collection.csv"), recursive=True)
    if not files:
        raise SystemExit(f"no *counter_collection.csv under {run_dir}")
    out = {}
    for fn in files:
        with open(fn) as f:
            for r in csv.DictReader(f):
                if r["Counter_Name"] != counter:
                    continue
                key = (fn, int(r["Dispatch_Id"]))
                name, v = out.get(key, (r["Kernel_Name"], 0.0))
                out[key] = (name, v + float(r["Counter_Value"]))
    return out


def summarize_traffic(args):
    """HBM bytes per partial-kernel launch from FETCH_SIZE and WRITE_SIZE runs of --profile-only.

    Both counters are read in KiB per dispatch. Each is scaled by what it reads for the calibration
    copy (CALIB_BYTES read and CALIB_BYTES written per launch, the last CALIB_COPIES dispatches)."""
    res = {}
    for counter, run_dir in (("FETCH_SIZE", args.traffic_summary[0]), ("WRITE_SIZE", args.traffic_summary[1])):
        d = _pmc_dispatches(run_dir, counter)
        order = sorted(d)
        part = [d[k][1] for k in order if args.traffic_kernel in d[k][0]]
        other = [d[k][1] for k in order if not d[k][0].startswith("pd_")]
        calib = other[-CALIB_COPIES:]
        if not part or len(calib) < CALIB_COPIES:
            raise SystemExit(f"{counter}: {len(part)} {args.traffic_kernel} dispatches, {len(calib)} calibration copies")
        part.sort()
        calib.sort()
        p_kib, c_kib = part[len(part) // 2], calib[len(calib) // 2]
        factor = (CALIB_BYTES / 1024.0) / c_kib
        res[counter] = {"partial_kib_median": p_kib, "calib_copy_kib_median": c_kib, "calib_factor": factor,
                        "partial_bytes": p_kib * 1024.0 * factor, "dispatches": len(part)}
    total = res["FETCH_SIZE"]["partial_bytes"] + res["WRITE_SIZE"]["partial_bytes"]
    if args.traffic_kernel == "partial":
        what = {"kernel": "decode partial kernel", "workload": "MTP verify 4 x 24/4 heads, ctx 61440+4, bs 16",
                "nsplit": args.nsplit}
    else:
        what = {"kernel": args.traffic_kernel, "workload": args.traffic_workload}
    summary = {**what, "hbm_bytes_per_launch": round(total), "counters": res,
               "calibration": f"{CALIB_COPIES} copies of {CALIB_BYTES} bytes (read + write) after the partial "
                              f"launches; factor = known bytes / counter bytes"}
    with open(args.traffic_out, "w") as f:
        json.dump(summary, f, indent=1)
    print(json.dumps(summary))


COUNTERS = ("SQ_INSTS_VALU", "SQ_INSTS_SALU", "SQ_INSTS_LDS", "SQ_INSTS_MFMA", "SQ_WAVES", "SQ_BUSY_CU_CYCLES",
            "SQ_VALU_MFMA_BUSY_CYCLES", "GRBM_GUI_ACTIVE")


def summarize_counters(args):
    """Instruction mix and MFMA utilisation per kernel launch from one rocprofv3 --pmc run with
    COUNTERS (medians over the dispatches), per wave and per 32-key tile: the decode partial kernel
    of --profile-only (--counters-kernel partial; a tile is one wave's 32 keys) or the config-5
    prefill kernel of --profile-prefill (--counters-kernel prefill, the 256-row kernel; a tile is 32
    keys that every wave of a workgroup computes for its 64 rows, counted once per wave)."""
    kind = args.counters_kernel
    per = {c: _pmc_dispatches(args.counters_summary, c) for c in COUNTERS}
    med = {}
    for c, d in per.items():
        v = sorted(x for name, x in d.values() if kind in name and "combine" not in name)
        if not v:
            raise SystemExit(f"{c}: no {kind}-kernel dispatches")
        med[c] = v[len(v) // 2]
    import workload as wl

    if kind == "partial":
        case = decode_case(wl, 2)
        tiles = 4 * (((case.seq_lens[0].item() - 1) // 32) + 1)  # 32-key tiles over the 4 kv heads
        what = {"kernel": "decode partial kernel", "workload": "MTP verify 4 x 24/4 heads, ctx 61440+4, bs 16",
                "nsplit": args.nsplit}
    else:
        # workgroup q of a kv head: rows (token x 6 heads) [256 q, 256 q + 256) of the chunk, keys up to the
        # last row's token; the key splits share these tiles
        tiles = 4 * sum(-(-(PREFILL_CTX + (256 * q + 255) // 6 + 1) // 32) for q in range(PREFILL_CHUNK * 6 // 256))
        tiles *= 4  # each of the 4 waves computes every tile of its workgroup
        what = {"kernel": "chunked prefill kernel", "workload": DESCRIPTIONS[5]}
    waves = med["SQ_WAVES"]
    simd_cycles = med["SQ_BUSY_CU_CYCLES"] / 256 * 1.0  # per CU: 4 SIMDs, each busy that long
    summary = {
        **what, "counters_median_per_dispatch": {c: round(v) for c, v in med.items()},
        "per_wave": {c: round(med[c] / waves, 1) for c in ("SQ_INSTS_VALU", "SQ_INSTS_SALU", "SQ_INSTS_LDS", "SQ_INSTS_MFMA")},
        "per_tile": {c: round(med[c] / tiles, 1) for c in ("SQ_INSTS_VALU", "SQ_INSTS_SALU", "SQ_INSTS_LDS", "SQ_INSTS_MFMA")},
        "tiles": tiles,
        "mfma_busy": round(med["SQ_VALU_MFMA_BUSY_CYCLES"] / (4 * 256 * simd_cycles), 4),
        "note": "SQ_INSTS_VALU includes the MFMA instructions; mfma_busy = SQ_VALU_MFMA_BUSY_CYCLES / "
                "(1024 SIMDs x SQ_BUSY_CU_CYCLES / 256 CUs)",
    }
    with open(args.counters_out, "w") as f:
        json.dump(summary, f, indent=1)
    print(json.dumps(summary))


def calibration_copies(torch, dev):
    """CALIB_COPIES plain copies of CALIB_BYTES (read and written once each): the known sizes the
    rocprofv3 FETCH_SIZE / WRITE_SIZE readings are scaled by."""
    src = torch.ones(CALIB_BYTES // 4, dtype=torch.float32, device=dev)
    dst = torch.empty_like(src)
    torch.cuda.synchronize()
    for _ in range(CALIB_COPIES):
        dst.copy_(src)
    torch.cuda.synchronize()


def load_package():
    import importlib.util

    if "mi50_vllm_lab_amd" in sys.modules:
        return sys.modules["mi50_vllm_lab_amd"]
    spec = importlib.util.spec_from_file_location("mi50_vllm_lab_amd", os.path.join(PKG_DIR, "__init__.py"),
                                                  submodule_search_locations=[PKG_DIR])
    mod = importlib.util.module_from_spec(spec)
    sys.modules["mi50_vllm_lab_amd"] = mod
    spec.loader.exec_module(mod)
    return mod


def cpu_model() -> str:
    try:
        out = subprocess.run(["lscpu"], capture_output=True, text=True, timeout=10).stdout
        for line in out.splitlines():
            if line.startswith("Model name"):
                return line.split(":", 1)[1].strip()
    except Exception:
        pass
    return platform.processor() or "unknown"


def decode_case(wl, n):
    """The decode workloads (seed 1000 + config number)."""
    s = 1000 + n
    if n == 1:
        return wl.make_case([4096], [1], num_q_heads=24, num_kv_heads=4, block_size=16, seed=s)
    if n == 2:
        return wl.make_case([61440], [4], num_q_heads=24, num_kv_heads=4, block_size=16, seed=s)
    if n == 3:
        return wl.make_case([2048, 9216, 33792, 122880], [8, 8, 8, 8], num_q_heads=24, num_kv_heads=4,
                            block_size=16, seed=s, causal=False, window=2048, poison=True)
    if n == 4:
        return wl.make_case([200000], [4], num_q_heads=24, num_kv_heads=4, block_size=16, seed=s,
                            outlier_frac=0.01, outlier_mult=50.0)
    raise ValueError(n)


DESCRIPTIONS = {
    1: "single-token decode: 1 seq x 1 query token, 24 q / 4 kv heads, ctx 4096+1, bs 16",
    2: "MTP verify decode: 1 seq x 4 query tokens, 24 q / 4 kv heads, head_dim 256, ctx 61440+4 int8 "
       "per-token-head paged KV, block_size 16",
    3: "DFlash2 drafter decode: 4 seqs (ctx 2048/9216/33792/122880) x 8 non-causal query tokens, 2048-key "
       "sliding window, freed pages NaN, 24 q / 4 kv heads, bs 16",
    4: "long-context decode: 1 seq x 4 query tokens, ctx 200000+4, 1% outlier rows x50, bs 16, one call "
       "captured in a HIP graph and replayed 1000x",
    5: "chunked prefill: 1 seq, 2048-token causal chunk over 61440 cached tokens (63488 keys), 24 q / 4 kv "
       "heads, head_dim 256, int8 per-token-head paged KV, bs 16",
}


def graph_of(torch, stream, calls):
    """A HIP graph holding `calls` (a list of zero-argument launch functions), captured on `stream`."""
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        for fn in calls:
            fn()
    return g


def time_replays(torch, graph, replays, stream):
    """ms for `replays` back-to-back replays of `graph`: HIP events on `stream`, device
    synchronisation on both sides."""
    torch.cuda.synchronize()
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record(stream)
    for _ in range(replays):
        graph.replay()
    end.record(stream)
    torch.cuda.synchronize()
    return start.elapsed_time(end)


class DecodeBench:
    """A decode workload on the device: rotating cache copies, output and segment buffers, and the
    operator call / partial-kernel call on a given copy."""

    def __init__(self, torch, wl, pd, dev, case, copies, nsplit):
        self.case = case
        self.d = d = case.to(dev)
        self.caches = [d.cache] + [wl.clone_cache(d.cache) for _ in range(copies - 1)]
        T, HQ = d.num_tokens, d.num_q_heads
        self.out = torch.empty((T, HQ, 256), dtype=torch.float16, device=dev)
        self.po, self.pm, self.pl = wl.partial_buffers(T, HQ, NSEG, dev)
        self.nsplit = nsplit
        self.pd = pd
        self.alg_bytes = wl.algorithmic_bytes(case)
        # the partial pass writes no output rows
        self.partial_bytes = self.alg_bytes - 2 * T * HQ * 256
        self.flops = wl.algorithmic_flops(case)

    def op(self, i):
        d, c = self.d, self.caches[i % len(self.caches)]
        return lambda: self.pd.decode(d.q, c.key_cache, c.value_cache, c.k_scale, c.v_scale, d.block_table,
                                      d.seq_lens, d.query_start_loc, self.out, d.scale, self.po, self.pm, self.pl,
                                      d.num_seqs, d.qmax, self.nsplit, d.window, d.causal)

    def partial(self, i):
        d, c = self.d, self.caches[i % len(self.caches)]

        def run():
            rc = self.pd.launch_partial(d.q, c.key_cache, d.block_table, d.seq_lens, d.query_start_loc, self.po,
                                        self.pm, self.pl, num_seqs=d.num_seqs, heads_q=d.num_q_heads,
                                        heads_kv=c.num_kv_heads, block_size=c.block_size, scale=d.scale,
                                        qmax=d.qmax, nsplit=self.nsplit, window=d.window, causal=d.causal)
            if rc != 0:
                raise RuntimeError(f"pth_dec_launch_partial failed: {rc}")
        return run


def cpu_decode_baseline(orc, case, runs, what):
    """Median seconds of the float64 oracle on the whole layer (after one warm-up)."""
    import numpy as np

    def once():
        orc.paged_decode(case.q, case.cache.key_cache, case.cache.value_cache, case.cache.k_scale,
                         case.cache.v_scale, case.block_table, case.seq_lens, case.query_start_loc, case.num_seqs,
                         case.scale, case.window, case.causal)

    once()
    times = []
    for _ in range(runs):
        t0 = time.perf_counter()
        once()
        times.append(time.perf_counter() - t0)
    med = float(np.median(times))
    return med, (f"float64 numpy oracle (oracle/attention.py) on the full {what} layer (all 24 heads), median of "
                 f"{runs} runs after 1 warm-up, numpy/BLAS threads on {os.cpu_count()} cores ({cpu_model()})")


def decode_line(us, db):
    gbs = db.alg_bytes / (us * 1e-6) / 1e9
    return {"us_per_layer": round(us, 3), "GB_s": round(gbs, 1), "frac": round(gbs / HBM_PEAK_GBS, 4),
            "algorithmic_bytes": db.alg_bytes, "nsplit": db.nsplit,
            "tflops": round(db.flops / (us * 1e-6) / 1e12, 2)}


# kernels/pth_dec/test_dec.py:150-165: (B, q_len) x ctx, cells with B * ctx > 270,000 skipped
GRID = ((1, 4), (2, 4), (4, 4), (1, 1), (2, 1))
GRID_CTX = (4096, 16384, 32768, 65536, 131072)


def bench_grid(torch, wl, pd, shim, dev, stream, hq, hkv, block_size):
    """The reference's decode speed grid at hq / hkv heads and the given block size: µs per layer
    (whole operator) at the split count the vLLM shim picks and at 64, the reference's default.
    Each cell cycles enough cache copies (>= 512 MiB) that every call reads its KV from HBM, not
    from the 256 MB Infinity Cache; one line of JSON per cell."""
    rows = []
    for B, ql in GRID:
        for ctx in GRID_CTX:
            if B * ctx > 270000:
                continue
            c = wl.make_case([ctx] * B, [ql] * B, num_q_heads=hq, num_kv_heads=hkv, block_size=block_size, seed=1)
            copies = max(2, min(64, -(-(512 << 20) // c.cache.nbytes())))
            pick = shim.decode_splits(NSEG, -1, hkv, B, dev, c.seq_lens.tolist(), ql, hq)
            cell = {"B": B, "q_len": ql, "ctx": ctx, "heads": f"{hq}/{hkv}", "block_size": block_size,
                    "nsplit_pick": pick, "copies": copies}
            for ns in sorted({pick, 64}):
                db = DecodeBench(torch, wl, pd, dev, c, copies, ns)
                with torch.cuda.stream(stream):
                    for i in range(copies):
                        db.op(i)()
                torch.cuda.synchronize()
                g = graph_of(torch, stream, [db.op(i) for i in range(copies)])
                reps = max(3, 2000 // copies)
                with torch.cuda.stream(stream):
                    g.replay()
                    ms = time_replays(torch, g, reps, stream)
                us = ms * 1e3 / (reps * copies)
                cell[f"us_ns{ns}"] = round(us, 2)
                if ns == pick:
                    cell["GB_s"] = round(db.alg_bytes / (us * 1e-6) / 1e9, 1)
                del db, g
                torch.cuda.empty_cache()
            print(json.dumps(cell), flush=True)
            rows.append(cell)
            del c
    return rows


def committed_profile(name):
    p = os.path.join(PROFILES, name)
    if not os.path.exists(p):
        return None
    try:
        with open(p) as f:
            return json.load(f)
    except Exception:
        return None


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=2000, help="timed operator calls (config 2)")
    ap.add_argument("--warmup", type=int, default=200, help="untimed operator calls before them")
    ap.add_argument("--nsplit", type=int, default=64, help="config 2 split count")
    ap.add_argument("--rotate", type=int, default=8, help="distinct config-2 KV caches cycled through")
    ap.add_argument("--configs", default="1,3,4,5,w",
                    help="other configs to measure, 'w' for the KV-cache writer ('' for none)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--cpu-runs", type=int, default=5)
    ap.add_argument("--profile-only", action="store_true",
                    help="replay the config-2 partial kernel only (--steps launches), then plain copies of known "
                         "size that calibrate the rocprofv3 FETCH_SIZE / WRITE_SIZE counters")
    ap.add_argument("--traffic-summary", nargs=2, metavar=("FETCH_DIR", "WRITE_DIR"),
                    help="no GPU work: turn two rocprofv3 --pmc runs of --profile-only (FETCH_SIZE, WRITE_SIZE) "
                         "into HBM bytes per partial launch, written to --traffic-out")
    ap.add_argument("--traffic-out", default=os.path.join(PROFILES, "pd_partial_mtp61k_traffic.json"))
    ap.add_argument("--traffic-kernel", default="partial",
                    help="substring of the kernel name whose dispatches --traffic-summary reads")
    ap.add_argument("--traffic-workload", default="", help="workload description for --traffic-summary")
    ap.add_argument("--profile-prefill", type=int, default=0, metavar="N",
                    help="run N config-5 prefill chunks (alternating two cache copies) and nothing else, for "
                         "rocprofv3")
    ap.add_argument("--profile-prefill-chunk", type=int, default=0, metavar="TOKENS",
                    help="with --profile-prefill N: a chunk of TOKENS over the same 61,440 cached tokens through "
                         "forward_pth's key split (N + 4 calls, then 6 unsplit ones), instead of the 2,048-token chunk")
    ap.add_argument("--profile-kvwrite", type=int, default=0, metavar="N",
                    help="run N KV-cache writer calls on the largest writer workload and nothing else, for "
                         "rocprofv3")
    ap.add_argument("--counters-summary", metavar="PMC_DIR",
                    help="no GPU work: turn a rocprofv3 --pmc run of --profile-only with the counters in "
                         "bench.COUNTERS into instruction mix and MFMA utilisation, written to --counters-out")
    ap.add_argument("--counters-out", default=None,
                    help="default: profiles/pd_partial_mtp61k_counters.json (partial) or "
                         "profiles/pd_prefill_chunk2048_ctx61440_counters.json (prefill)")
    ap.add_argument("--counters-kernel", default="partial", choices=("partial", "prefill"))
    ap.add_argument("--prefill-grid", metavar="HQ,HKV,BS",
                    help="the reference's prefill sweep: one 2,048-token chunk over 0/16k/64k/128k cached tokens "
                         "(one JSON line per cell), e.g. 12,2,1584 (one TP=2 rank, as the reference) or 24,4,16")
    ap.add_argument("--grid", metavar="HQ,HKV,BS",
                    help="only the reference's decode speed grid (B x q_len x ctx) at HQ q heads, HKV kv heads "
                         "and block size BS, one JSON line per cell")
    args = ap.parse_args()

    if args.traffic_summary:
        summarize_traffic(args)
        return
    if args.counters_summary:
        if args.counters_out is None:
            args.counters_out = os.path.join(PROFILES, "pd_partial_mtp61k_counters.json" if args.counters_kernel ==
                                             "partial" else "pd_prefill_chunk2048_ctx61440_counters.json")
        summarize_counters(args)
        return

    if args.gpus != 1:
        print(json.dumps({"error": f"--gpus {args.gpus}: this benchmark measures one GPU; the operators are "
                                   "single-GPU (a multi-GPU deployment shards them by kv head) and no multi-GPU "
                                   "run is part of this build"}))
        sys.exit(2)

    import torch

    import workload as wl

    pkg = load_package()
    pd = pkg.pth_dec
    pd.load_library()
    if not torch.cuda.is_available():
        print(json.dumps({"error": "no GPU visible"}))
        sys.exit(1)
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    stream = torch.cuda.Stream()

    if args.prefill_grid:
        hq, hkv, bs = (int(x) for x in args.prefill_grid.split(","))
        bench_prefill_grid(torch, wl, pd, dev, stream, hq, hkv, bs)
        return

    if args.grid:
        hq, hkv, bs = (int(x) for x in args.grid.split(","))
        bench_grid(torch, wl, pd, pkg.vllm_shim, dev, stream, hq, hkv, bs)
        return

    if args.profile_kvwrite:
        res = bench_cache_write(torch, wl, pd, dev, stream, KVW_TOKENS[-1], reps=1, calls=args.profile_kvwrite)
        calibration_copies(torch, dev)
        print(json.dumps({"profile_kvwrite": True, "tokens": KVW_TOKENS[-1], "us_per_call": res["us_per_call"],
                          "GB_s": res["GB_s"], "calib_copies": CALIB_COPIES, "calib_bytes": CALIB_BYTES}))
        return

    if args.profile_prefill and args.profile_prefill_chunk:
        n = 2 * max(1, args.profile_prefill // 2)
        res = bench_short_prefill(torch, wl, pd, dev, stream, args.profile_prefill_chunk, reps=n)
        print(json.dumps({"profile_prefill": True, "tokens": res["tokens"], "nsplit": res["nsplit"],
                          "split_calls": n + 4, "ms_per_chunk": res["ms_per_chunk"], "ms_unsplit": res["ms_unsplit"]}))
        return

    if args.profile_prefill:
        res = bench_prefill(torch, wl, pd, dev, stream, reps=2 * max(1, args.profile_prefill // 2), exact_too=False)
        print(json.dumps({"profile_prefill": True, "chunks": 2 * max(1, args.profile_prefill // 2) + 4,
                          "ms_per_chunk": res["ms_per_chunk"]}))
        return

    case2 = decode_case(wl, 2)
    b2 = DecodeBench(torch, wl, pd, dev, case2, args.rotate, args.nsplit)
    R = len(b2.caches)
    with torch.cuda.stream(stream):  # eager warm-up of both paths on the side stream
        for i in range(R):
            b2.op(i)()
            b2.partial(i)()
    torch.cuda.synchronize()

    if args.profile_only:
        g = graph_of(torch, stream, [b2.partial(i) for i in range(args.steps)])
        with torch.cuda.stream(stream):
            g.replay()
        torch.cuda.synchronize()
        calibration_copies(torch, dev)
        print(json.dumps({"profile_only": True, "partial_launches": args.steps, "nsplit": args.nsplit,
                          "calib_copies": CALIB_COPIES, "calib_bytes": CALIB_BYTES}))
        return

    steps, warmup = max(1, args.steps), max(0, args.warmup)
    g_steps = graph_of(torch, stream, [b2.op(i) for i in range(steps)])
    g_warm = graph_of(torch, stream, [b2.op(i) for i in range(warmup)]) if warmup else None
    g_roof = graph_of(torch, stream, [b2.partial(i) for i in range(ROOF_LAUNCHES)])
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        if g_warm is not None:
            g_warm.replay()
        ms_total = time_replays(torch, g_steps, 1, stream)
        g_roof.replay()  # warm
        roof_ms = time_replays(torch, g_roof, 1, stream) / ROOF_LAUNCHES
    ms_step = ms_total / steps
    us_layer = ms_step * 1e3
    gbs = b2.alg_bytes / (ms_step * 1e-3) / 1e9
    part_gbs = b2.partial_bytes / (roof_ms * 1e-3) / 1e9

    traffic_j = committed_profile("pd_partial_mtp61k_traffic.json")
    traffic = traffic_j.get("hbm_bytes_per_launch") if traffic_j and traffic_j.get("nsplit") == args.nsplit else None
    counters = committed_profile("pd_partial_mtp61k_counters.json")

    want = [int(x) for x in args.configs.split(",") if x.strip().isdigit()]
    want_kvw = "w" in [x.strip() for x in args.configs.split(",")]
    configs = {}
    shim = pkg.vllm_shim
    for n in (1, 3, 4):
        if n not in want:
            continue
        c = decode_case(wl, n)
        ns = shim.decode_splits(NSEG, c.window, 4, c.num_seqs, dev, c.seq_lens.tolist(), c.qmax)
        # enough cache copies that the visible pages in rotation exceed the 256 MB Infinity Cache
        # (config 1: 32 x 8.5 MB; config 3: 16 x 17.1 MB); config 4 reads 416 MB per call
        copies = {1: 32, 3: 16, 4: 1}[n]
        db = DecodeBench(torch, wl, pd, dev, c, copies, ns)
        with torch.cuda.stream(stream):
            for i in range(copies):
                db.op(i)()
        torch.cuda.synchronize()
        if n == 4:
            g = graph_of(torch, stream, [db.op(0)])
            reps, per = 1000, 1
        else:
            g = graph_of(torch, stream, [db.op(i) for i in range(copies)])
            reps, per = (30 if n == 1 else 60), copies
        with torch.cuda.stream(stream):
            for _ in range(max(1, reps // 10)):
                g.replay()
            ms = time_replays(torch, g, reps, stream)
        us = ms * 1e3 / (reps * per)
        line = decode_line(us, db)
        line["workload"] = DESCRIPTIONS[n]
        line["timed"] = f"{reps} replays of a {per}-call graph" + (
            "" if n == 4 else f" over {copies} cache copies ({copies * wl.visible_kv_bytes(c) / 1e6:.0f} MB of "
                              f"visible pages in rotation)")
        configs[str(n)] = line
        del db, g
        torch.cuda.empty_cache()
    if 5 in want:
        configs["5"] = bench_prefill(torch, wl, pd, dev, stream)
    if want_kvw:
        configs["kv_write"] = {str(T): bench_cache_write(torch, wl, pd, dev, stream, T) for T in KVW_TOKENS}

    cpu = None
    if not args.no_cpu_baseline:
        from oracle import attention as orc

        med, sample = cpu_decode_baseline(orc, case2, args.cpu_runs, "config-2")
        cpu = {"value": round(b2.alg_bytes / med / 1e9, 4), "unit": "GB/s", "cores": os.cpu_count(), "kind": "port",
               "us_per_layer": round(med * 1e6, 1), "sample": sample, "gpu_speedup": round(med * 1e6 / us_layer, 1)}
        for n in (1, 4):
            if str(n) in configs:
                c = decode_case(wl, n)
                m, s = cpu_decode_baseline(orc, c, args.cpu_runs, f"config-{n}")
                configs[str(n)]["cpu_baseline"] = {
                    "us_per_layer": round(m * 1e6, 1), "GB_s": round(wl.algorithmic_bytes(c) / m / 1e9, 4),
                    "cores": os.cpu_count(), "kind": "port", "sample": s,
                    "gpu_speedup": round(m * 1e6 / configs[str(n)]["us_per_layer"], 1)}
        if "5" in configs:
            configs["5"]["cpu_baseline"] = cpu_prefill_baseline(torch, wl, orc)

    roofline = {"bound": "hbm", "achieved": round(part_gbs, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": round(part_gbs / HBM_PEAK_GBS, 4), "traffic": traffic, "kernel": pd.partial_kernel_name(24, 16),
                "avg_launch_us": round(roof_ms * 1e3, 3), "launches": ROOF_LAUNCHES,
                "bytes_per_launch": b2.partial_bytes}
    if counters:
        roofline["mfma_busy"] = counters.get("mfma_busy")
        roofline["counters_from"] = "profiles/pd_partial_mtp61k_counters.json"
    line = {
        "metric": METRIC,
        "value": round(gbs, 1),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": steps,
        "warmup": warmup,
        "ms_per_step": round(ms_step, 6),
        "us_per_layer": round(us_layer, 3),
        "pct_hbm_peak": round(100.0 * gbs / HBM_PEAK_GBS, 2),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "int8 KV / fp16 MFMA / fp32 softmax",
        "data": "synthetic (seeded N(0,1) K/V quantised absmax/127, random page permutation)",
        "config": {"workload": DESCRIPTIONS[2], "nsplit": args.nsplit, "rotating_caches": R,
                   "algorithmic_bytes": b2.alg_bytes, "kv_bytes": wl.visible_kv_bytes(case2), "flops": b2.flops,
                   "timed": f"one replay of a {steps}-call graph"},
        "roofline": roofline,
        "tflops": round(b2.flops / (ms_step * 1e-3) / 1e12, 2),
        "cpu_baseline": cpu,
        "configs": configs,
    }
    print(json.dumps(line))


PREFILL_CTX, PREFILL_CHUNK = 61440, 2048


def bench_prefill(torch, wl, pd, dev, stream, reps=20, exact_too=True):
    """Config 5: ms per chunk and TFLOP/s of the chunked-prefill operator (pth_fa_forward), and
    of pth_fa_forward_exact on the same chunk under `exact`."""
    ctx, sq = PREFILL_CTX, PREFILL_CHUNK
    case = wl.make_case([ctx], [sq], num_q_heads=24, num_kv_heads=4, block_size=16, seed=1005)
    flops = wl.prefill_flops([ctx + sq], [ctx], sq, 24)
    d = case.to(dev)
    caches = [d.cache, wl.clone_cache(d.cache)]
    q = wl.prefill_query(d)
    qa = torch.tensor([ctx], dtype=torch.int32, device=dev)
    out = torch.empty((1, sq, 24, 256), dtype=torch.float32, device=dev)

    def op(c, exact=False):
        return lambda: pd.forward_pth(q, c.key_cache, c.value_cache, d.block_table, d.seq_lens, d.scale, qa, out=out,
                                      exact=exact)

    def timed(exact):
        with torch.cuda.stream(stream):
            for c in caches:
                op(c, exact)()
        torch.cuda.synchronize()
        g = graph_of(torch, stream, [op(c, exact) for c in caches])
        with torch.cuda.stream(stream):
            g.replay()
            return time_replays(torch, g, reps // 2, stream) / reps

    ms = timed(False)
    tflops = flops / (ms * 1e-3) / 1e12
    line = {"workload": DESCRIPTIONS[5], "ms_per_chunk": round(ms, 4), "TFLOP_s": round(tflops, 1),
            "frac": round(tflops / MFMA_FP16_PEAK_TFLOPS, 4), "flops": flops, "peak": MFMA_FP16_PEAK_TFLOPS,
            "bound": "mfma", "timed": f"{reps // 2} replays of a 2-call graph over 2 cache copies"}
    ctr = committed_profile("pd_prefill_chunk2048_ctx61440_counters.json")
    if ctr:
        line["mfma_busy"] = ctr.get("mfma_busy")
        line["per_tile"] = ctr.get("per_tile")
        line["counters_from"] = "profiles/pd_prefill_chunk2048_ctx61440_counters.json"
    if exact_too:
        mse = timed(True)
        tfe = flops / (mse * 1e-3) / 1e12
        line["exact"] = {"entry": "pth_fa_forward_exact", "ms_per_chunk": round(mse, 4), "TFLOP_s": round(tfe, 1),
                         "frac": round(tfe / MFMA_FP16_PEAK_TFLOPS, 4)}
        line["chunk64"] = bench_short_prefill(torch, wl, pd, dev, stream, 64)
        line["chunk2560"] = bench_short_prefill(torch, wl, pd, dev, stream, 2560, reps=10)
    return line


def bench_short_prefill(torch, wl, pd, dev, stream, sq, reps=200):
    """A chunk of sq tokens over the same 61,440 cached tokens, with the key split that forward_pth
    picks (0: dealt evenly, pth_fa_forward_balanced): 64 tokens give too few query tiles to fill the
    GPU, 2,560 give 320 workgroups of 192 rows (two rounds) or 240 of 256 rows (one)."""
    ctx = PREFILL_CTX
    case = wl.make_case([ctx], [sq], num_q_heads=24, num_kv_heads=4, block_size=16, seed=1005)
    flops = wl.prefill_flops([ctx + sq], [ctx], sq, 24)
    d = case.to(dev)
    caches = [d.cache, wl.clone_cache(d.cache)]
    q = wl.prefill_query(d)
    qa = torch.tensor([ctx], dtype=torch.int32, device=dev)
    out = torch.empty((1, sq, 24, 256), dtype=torch.float32, device=dev)
    keys = d.block_table.shape[1] * 16
    nsplit = pd._prefill_plan(1, sq, 24, 4, keys, 16, sq)

    def timed(ns, n):
        ops = [lambda c=c: pd.forward_pth(q, c.key_cache, c.value_cache, d.block_table, d.seq_lens, d.scale, qa,
                                          out=out, nsplit=ns, max_keys=keys) for c in caches]
        with torch.cuda.stream(stream):
            for o in ops:
                o()
        torch.cuda.synchronize()
        g = graph_of(torch, stream, ops)
        with torch.cuda.stream(stream):
            g.replay()
            return time_replays(torch, g, n // 2, stream) / n

    ms = timed(None, reps)
    ms1 = timed(1, max(2, reps // 20))
    kv = (ctx + sq) * 4 * 520
    return {"tokens": sq, "nsplit": nsplit, "ms_per_chunk": round(ms, 4),
            "TFLOP_s": round(flops / (ms * 1e-3) / 1e12, 1), "KV_GB_s": round(kv / (ms * 1e-3) / 1e9, 1),
            "ms_unsplit": round(ms1, 4), "timed": f"{reps // 2} replays of a 2-call graph over 2 cache copies"}


PREFILL_GRID_CTX = (0, 16384, 65536, 131072)
# kernels/fa_pth/test_pth.py:113-125 on MI50, one TP=2 rank (12 q / 2 kv heads, block size 1,584):
# ms per 2,048-token chunk over each cached context (docs/logs/test_pth.log:11-14)
PREFILL_GRID_MI50_MS = {0: 7.2, 16384: 98.2, 65536: 376.2, 131072: 747.4}


def bench_prefill_grid(torch, wl, pd, dev, stream, hq, hkv, block_size, reps=20):
    """The reference's prefill speed sweep (kernels/fa_pth/test_pth.py:113-125): one 2,048-token
    causal chunk on top of 0 / 16k / 64k / 128k cached tokens, through forward_pth with the key
    split it picks for the chunk's keys (max_keys = ctx + 2,048), timed as graph replays over two
    cache copies. FLOPs as test_pth.py:118, 4 D Hq (2048 ctx + 2048 * 2049 / 2). One JSON line per
    cell, with the unsplit time as well."""
    sq = PREFILL_CHUNK
    for ctx in PREFILL_GRID_CTX:
        case = wl.make_case([ctx], [sq], num_q_heads=hq, num_kv_heads=hkv, block_size=block_size, seed=1500 + ctx % 997)
        d = case.to(dev)
        caches = [d.cache, wl.clone_cache(d.cache)]
        q = wl.prefill_query(d)
        qa = torch.tensor([ctx], dtype=torch.int32, device=dev)
        out = torch.empty((1, sq, hq, 256), dtype=torch.float32, device=dev)
        flops = 4 * 256 * hq * (sq * ctx + sq * (sq + 1) // 2)
        pick = pd._prefill_plan(1, sq, hq, hkv, ctx + sq, block_size, sq)

        def timed(ns, n):
            ops = [lambda c=c: pd.forward_pth(q, c.key_cache, c.value_cache, d.block_table, d.seq_lens, d.scale, qa,
                                              out=out, nsplit=ns, max_keys=ctx + sq) for c in caches]
            with torch.cuda.stream(stream):
                for o in ops:
                    o()
            torch.cuda.synchronize()
            g = graph_of(torch, stream, ops)
            with torch.cuda.stream(stream):
                g.replay()
                return time_replays(torch, g, n // 2, stream) / n

        n = reps if ctx <= 65536 else max(4, reps // 2)
        ms = timed(None, n)
        ms1 = ms if pick == 1 else timed(1, n)
        mi50 = PREFILL_GRID_MI50_MS[ctx]
        print(json.dumps({"prefill_grid": True, "heads_q": hq, "heads_kv": hkv, "block_size": block_size,
                          "ctx": ctx, "chunk": sq, "nsplit_pick": pick, "ms_per_chunk": round(ms, 4),
                          "ms_unsplit": round(ms1, 4), "TFLOP_s": round(flops / (ms * 1e-3) / 1e12, 1),
                          "frac": round(flops / (ms * 1e-3) / 1e12 / MFMA_FP16_PEAK_TFLOPS, 4), "flops": flops,
                          "mi50_rank_ms": mi50, "timed": f"{n // 2} replays of a 2-call graph over 2 cache copies"}),
              flush=True)
        del caches, d, case, q, out
        torch.cuda.empty_cache()


KVW_TOKENS = (4, 2048, 32768)


def bench_cache_write(torch, wl, pd, dev, stream, T, reps=None, calls=None):
    """The KV-cache writer (pth_cache_write) on T new tokens of one sequence: key and value fp16
    [T, 4, 256] as the strided views vLLM hands over (slices of one fused QKV projection output
    [T, (24 + 2 x 4) x 256]), slots at positions 0..T-1 of a sequence whose 16-slot blocks are a
    random permutation of the cache's, HND layout. Inputs and caches rotate over enough copies that
    every call reads and writes HBM rather than the 256 MB Infinity Cache. Bytes: K and V read
    (2 x T x 4 x 512), the slot mapping (8 T), the rows written (T x 4 x 520)."""
    hq, hkv, D, bs = 24, 4, 256, 16
    read = 2 * T * hkv * D * 2 + 8 * T
    write = T * hkv * 520
    copies = max(2, min(64, -(-(512 << 20) // (read + write))))
    g = torch.Generator().manual_seed(77 + T)
    gd = torch.Generator(device=dev).manual_seed(77 + T)
    nblk = -(-T // bs)
    perm = torch.randperm(nblk, generator=g)
    pos = torch.arange(T)
    slots = (perm[pos // bs] * bs + pos % bs).to(torch.int64).to(dev)
    qkvs, caches = [], []
    for i in range(copies):
        qkvs.append(torch.randn((T, (hq + 2 * hkv) * D), generator=gd, device=dev, dtype=torch.float16))
        caches.append(wl.allocate_cache(nblk, bs, hkv, "HND", device=dev))

    def op(i):
        qkv, c = qkvs[i], caches[i]
        k = qkv[:, hq * D:(hq + hkv) * D].view(T, hkv, D)
        v = qkv[:, (hq + hkv) * D:].view(T, hkv, D)
        return lambda: pd.cache_write(k, v, c.key_cache, c.value_cache, c.k_scale, c.v_scale, slots)

    with torch.cuda.stream(stream):
        for i in range(copies):
            op(i)()
    torch.cuda.synchronize()
    per = calls or copies
    gr = graph_of(torch, stream, [op(i % copies) for i in range(per)])
    reps = reps or max(3, 4000 // per)
    with torch.cuda.stream(stream):
        gr.replay()
        ms = time_replays(torch, gr, reps, stream)
    us = ms * 1e3 / (reps * per)
    gbs = (read + write) / (us * 1e-6) / 1e9
    del gr, qkvs, caches
    torch.cuda.empty_cache()
    return {"tokens": T, "us_per_call": round(us, 3), "GB_s": round(gbs, 1), "frac": round(gbs / HBM_PEAK_GBS, 4),
            "algorithmic_bytes": read + write,
            "workload": f"KV-cache writer: {T} tokens x 4 kv heads, fp16 K/V as strided views of a fused QKV "
                        f"buffer, random 16-slot pages, HND",
            "timed": f"{reps} replays of a {per}-call graph over {copies} input/cache copies"}


def cpu_prefill_baseline(torch, wl, orc, nrows=24):
    import numpy as np

    ctx, sq = PREFILL_CTX, PREFILL_CHUNK
    case = wl.make_case([ctx], [sq], num_q_heads=24, num_kv_heads=4, block_size=16, seed=1005)
    flops = wl.prefill_flops([ctx + sq], [ctx], sq, 24)
    rows = np.linspace(0, sq - 1, nrows).astype(int).tolist()
    qcpu = wl.prefill_query(case)
    qa_cpu = torch.tensor([ctx], dtype=torch.int32)

    def once():
        orc.paged_prefill(qcpu, case.cache.key_cache, case.cache.value_cache, case.cache.k_scale, case.cache.v_scale,
                          case.block_table, case.seq_lens, case.scale, qa_cpu, rows)

    once()
    times = []
    for _ in range(3):
        t0 = time.perf_counter()
        once()
        times.append(time.perf_counter() - t0)
    med = float(np.median(times))
    sample_flops = 4 * 256 * 24 * sum(min(ctx + sq, ctx + r + 1) for r in rows)
    return {"TFLOP_s": round(sample_flops / med / 1e12, 6), "cores": os.cpu_count(), "kind": "port",
            "sample": f"float64 numpy oracle (oracle/attention.py paged_prefill) on {len(rows)} of the {sq} query "
                      f"rows (all 24 heads, full visible context each), median of 3 runs after 1 warm-up, BLAS "
                      f"threads on {os.cpu_count()} cores ({cpu_model()})",
            "est_ms_full_chunk": round(flops / (sample_flops / med) * 1e3, 1)}


if __name__ == "__main__":
    main()
