"""The work that a user of this library has it do, as measurable cases.

The library is one attention layer over vLLM's int8 per-token-head paged KV cache: the split-K
decode, the chunked prefill and the cache writer, called one by one or through the vLLM routing
shim. Sizes come from this repository's benchmark and tests: 24 q / 4 kv heads (the whole model on
one GPU) and 12 / 2 (one of two tensor-parallel ranks), head size 256, block sizes 16 and 1,584,
contexts up to 200,000 keys, 1 to 8 query tokens per decoded sequence, chunks of up to 2,048.

A case is a plain dict; `kind` says which entry points it takes:
  step   one decode step of `layers` layers as a serving engine runs it: per layer the cache writer
         stores the new tokens' K/V, then the shim routes the batch to the decode operator.
         `graph`: the step is captured once in a HIP graph and replayed, else called eagerly.
  decode one call of the decode operator (windowed and non-causal rows, long contexts).
  fa     one call of the chunked-prefill operator on one sequence.
  mixed  one layer of a mixed batch through the shim: decoded sequences, then prompt chunks.
  write  one call of the cache writer.
"""
import importlib.util
import math
import os
import random
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_DIM, _ROW = 256, 520
_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
_SCALE = 1.0 / math.sqrt(_DIM)


def _package():
    name = "mi50_vllm_lab_amd"
    if name not in sys.modules:
        d = os.path.join(_ROOT, "mi50-vllm-lab_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(d, "__init__.py"),
                                                      submodule_search_locations=[d])
        sys.modules[name] = mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
    return sys.modules[name]


def _case(name, kind, **kw):
    c = {"name": name, "kind": kind, "heads_q": 24, "heads_kv": 4, "block_size": 16, "layout": "HND", "outliers": 0.0}
    c.update(kw)
    return c


def listed():
    return [
        # one user, one new token, short context, no graph: launches and host work are what is left
        _case("step_1tok_4k_eager", "step", seqs=1, qlen=1, ctx_lo=4096, ctx_hi=4096, layers=1, graph=False, window=-1),
        # the benchmark's decode: multi-token verification of 4 tokens over a 61k context, graph-captured
        _case("step_mtp_61k_graph", "step", seqs=1, qlen=4, ctx_lo=61440, ctx_hi=61440, layers=4, graph=True, window=-1),
        # a serving batch of single-token rows with contexts of all lengths, graph-captured
        _case("step_batch48_graph", "step", seqs=48, qlen=1, ctx_lo=200, ctx_hi=16384, layers=4, graph=True, window=-1),
        # a smaller batch of verification rows at one rank's heads and the reference's block size, eager
        _case("step_batch13_mtp_eager", "step", seqs=13, qlen=4, ctx_lo=500, ctx_hi=32768, layers=2, graph=False,
              window=-1, heads_q=12, heads_kv=2, block_size=1584),
        # the drafter: 8 non-causal rows per sequence in a 2,048-key window, mixed contexts
        _case("decode_drafter_window", "decode", seqs=4, qlen=8, ctx_lo=2048, ctx_hi=122880, window=2048, causal=False),
        # long context with outlier tokens
        _case("decode_200k_outliers", "decode", seqs=1, qlen=4, ctx_lo=200000, ctx_hi=200000, window=-1, causal=True,
              outliers=0.01),
        # the benchmark's prompt chunk over a long cached context
        _case("fa_2048_ctx61k", "fa", tokens=2048, ctx=61440, exact=False),
        # the decode's numerics, one rank's heads, the reference's block size
        _case("fa_exact_2048_rank", "fa", tokens=2048, ctx=16384, exact=True, heads_q=12, heads_kv=2, block_size=1584),
        # the end of a prompt: a short ragged chunk over a long context
        _case("fa_77_ctx30k", "fa", tokens=77, ctx=30011, exact=False),
        # a fresh prompt of odd length through the shim
        _case("mixed_fresh_1501", "mixed", seqs=0, qlen=1, ctx_lo=0, ctx_hi=0, chunks=1, chunk_lo=1501, chunk_hi=1501,
              chunk_ctx=0),
        # a busy step: decoded sequences, then several prompt chunks of different lengths over cached prefixes
        _case("mixed_9dec_4chunks", "mixed", seqs=9, qlen=1, ctx_lo=300, ctx_hi=20000, chunks=4, chunk_lo=70,
              chunk_hi=900, chunk_ctx=6000),
        # a long prompt's K/V into the cache, bf16 views of a fused QKV buffer
        _case("write_32k_bf16", "write", tokens=32768, dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges; none costs more than fa_2048_ctx61k."""
    hq, hkv = rng.choice([(24, 4), (24, 4), (12, 2)])
    common = {"heads_q": hq, "heads_kv": hkv, "block_size": rng.choice([16, 16, 32, 1584]),
              "layout": rng.choice(["HND", "HND", "NHD"]), "outliers": rng.choice([0.0, 0.0, 0.01])}
    kind = rng.choice(["step", "step", "decode", "fa", "fa", "mixed", "write"])
    c = _case("", kind, **common)
    del c["name"]
    if kind == "step":
        seqs = _log_int(rng, 1, 64)
        hi = _log_int(rng, 300, min(131072, 800000 // seqs))
        c.update(seqs=seqs, qlen=rng.choice([1, 1, 2, 4]), ctx_lo=max(40, hi // rng.choice([1, 8, 64])), ctx_hi=hi,
                 layers=rng.choice([1, 2, 4]), graph=rng.random() < 0.5, window=-1)
        c["ctx_lo"] = min(c["ctx_lo"], c["ctx_hi"])
    elif kind == "decode":
        windowed = rng.random() < 0.5
        seqs = _log_int(rng, 1, 8)
        hi = _log_int(rng, 1000, 200000 // seqs)
        c.update(seqs=seqs, qlen=rng.choice([1, 3, 4, 5, 8]) if windowed else rng.choice([1, 2, 4]),
                 ctx_lo=max(60, hi // 4), ctx_hi=hi, window=rng.choice([512, 2048, 4096]) if windowed else -1,
                 causal=rng.random() < 0.3 if windowed else True)
    elif kind == "fa":
        tokens = _log_int(rng, 64, 2048)
        c.update(tokens=tokens, ctx=rng.choice([0, _log_int(rng, 100, 61440)]), exact=False)
        if rng.random() < 0.3:
            c.update(exact=True, ctx=min(c["ctx"], 32768))
    elif kind == "mixed":
        chunks = rng.choice([1, 1, 2, 4])
        hi = _log_int(rng, 80, 1600 // chunks + 100)
        c.update(seqs=rng.choice([0, 3, _log_int(rng, 4, 32)]), qlen=rng.choice([1, 4]), ctx_lo=100,
                 ctx_hi=_log_int(rng, 200, 16000), chunks=chunks, chunk_lo=max(64, hi // 3), chunk_hi=max(64, hi),
                 chunk_ctx=rng.choice([0, _log_int(rng, 50, 8000)]))
    else:
        c.update(tokens=_log_int(rng, 16, 32768), dtype=rng.choice(["fp16", "bf16", "fp32"]), outliers=0.0)
    return c


# ---- shapes: fixed by the case, so that work() knows them ----

def _spread(case, key, n, lo, hi):
    """n lengths between lo and hi, evenly spread over their logarithm, in an order fixed by the case."""
    if n <= 0:
        return []
    a, b = math.log(max(1, lo)), math.log(max(1, hi))
    out = [int(round(math.exp(a + (b - a) * (i + 0.5) / n))) for i in range(n)] if n > 1 else [hi]
    if n > 1:
        out[0], out[-1] = max(1, lo), max(1, hi)
    random.Random("%s %s %d %d" % (key, case["kind"], n, hi)).shuffle(out)
    return out


def _shape(case):
    """(cached tokens, new tokens) per sequence."""
    k = case["kind"]
    if k == "fa":
        return [case["ctx"]], [case["tokens"]]
    if k in ("step", "decode"):
        return _spread(case, "ctx", case["seqs"], case["ctx_lo"], case["ctx_hi"]), [case["qlen"]] * case["seqs"]
    ctx = _spread(case, "ctx", case["seqs"], case["ctx_lo"], case["ctx_hi"])
    new = _spread(case, "chunk", case["chunks"], case["chunk_lo"], case["chunk_hi"])
    pre = [case["chunk_ctx"] * (i + 1) // case["chunks"] for i in range(case["chunks"])]
    return ctx + pre, [case["qlen"]] * case["seqs"] + new


def _rand_rows(gen, rows, outliers):
    """int8 cache rows [rows, 520] of K, V ~ N(0, 1) (a share `outliers` of them times 50)."""
    kv = torch.empty((rows, _ROW), dtype=torch.int8, device="cuda")
    step = 1 << 17
    for r in range(0, rows, step):
        n = min(step, rows - r)
        x = torch.randn((n, 2, _DIM), device="cuda", generator=gen)
        if outliers:
            x *= torch.where(torch.rand((n, 2, 1), device="cuda", generator=gen) < outliers, 50.0, 1.0)
        s = x.abs().amax(-1, keepdim=True) / 127.0
        kv[r:r + n].view(n, 2, 260)[:, :, :_DIM] = (x / s).round_().clamp_(-127, 127).to(torch.int8)
        kv[r:r + n].view(n, 2, 260)[:, :, _DIM:] = s.view(torch.int8).view(n, 2, 4)
    return kv


def _inputs(case, seed):
    """Everything the case's call reads, from the seed alone: raw caches and metadata, no operator."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    host = torch.Generator().manual_seed(seed)
    hq, hkv, bs = case["heads_q"], case["heads_kv"], case["block_size"]
    x = {}
    if case["kind"] == "write":
        t, dt = case["tokens"], _DTYPES[case["dtype"]]
        x["qkv"] = torch.randn((t, (hq + 2 * hkv) * _DIM), device="cuda", generator=gen).to(dt)
        pages = -(-t // bs) + 2
        perm = torch.randperm(pages, generator=host)[: -(-t // bs)]
        slots = (perm[:, None] * bs + torch.arange(bs)[None, :]).reshape(-1)[:t]
        x["slots"], x["pages"] = slots.to("cuda", torch.int64), pages
        return x
    ctx, new = _shape(case)
    seqs = [c + n for c, n in zip(ctx, new)]
    per = [-(-s // bs) for s in seqs]
    pages = sum(per) + 2
    perm = torch.randperm(pages, generator=host).to(torch.int32)
    bt = torch.zeros((len(seqs), max(per) + 1), dtype=torch.int32)
    o = 0
    for b, n in enumerate(per):
        bt[b, :n] = perm[o:o + n]
        o += n
    layers = case.get("layers", 1)
    shape = (pages, hkv, bs, _ROW) if case["layout"] == "HND" else (pages, bs, hkv, _ROW)
    x["kv"] = [_rand_rows(gen, pages * bs * hkv, case["outliers"]).view(shape) for _ in range(layers)]
    x["kv"] = [k if case["layout"] == "HND" else k.transpose(1, 2) for k in x["kv"]]
    total = sum(new)
    x["q"] = [torch.randn((total, hq, _DIM), device="cuda", generator=gen).half() for _ in range(layers)]
    if case["kind"] == "step":
        x["new"] = [torch.randn((total, 2, hkv, _DIM), device="cuda", generator=gen).half() for _ in range(layers)]
        x["slots"] = torch.cat([bt[b].long()[torch.arange(c, s) // bs] * bs + torch.arange(c, s) % bs
                                for b, (c, s) in enumerate(zip(ctx, seqs))]).to("cuda")
    if case["kind"] == "fa":
        x["q"] = [q.float().transpose(0, 1).unsqueeze(0).contiguous() for q in x["q"]]
    x["bt"], x["lens_cpu"] = bt.to("cuda"), torch.tensor(seqs, dtype=torch.int32)
    x["lens"] = x["lens_cpu"].to("cuda")
    x["qsl_cpu"] = torch.tensor([0] + new).cumsum(0).to(torch.int32)
    x["qsl"] = x["qsl_cpu"].to("cuda")
    x["q_abs"] = torch.tensor(ctx, dtype=torch.int32, device="cuda")
    return x


def _segments(tokens, hq, nseg=64):
    return [torch.empty((tokens, hq, nseg) + d, dtype=torch.float32, device="cuda") for d in ((_DIM,), (), ())]


def prepare(case, seed):
    pkg = _package()
    x = _inputs(case, seed)
    hq, hkv, bs, kind = case["heads_q"], case["heads_kv"], case["block_size"], case["kind"]
    s = {"pkg": pkg, "case": case}
    if kind == "write":
        s["cache"] = pkg.kvcache.allocate_cache(x["pages"], bs, hkv, case["layout"], "cuda")
        kv = x["qkv"][:, hq * _DIM:].view(case["tokens"], 2, hkv, _DIM)
        s.update(qkv=x["qkv"], key=kv[:, 0], value=kv[:, 1], slots=x["slots"])
        return s
    s.update(x)
    s["caches"] = [pkg.kvcache.cache_views(k, case["layout"]) for k in x["kv"]]
    s["out"] = [torch.zeros_like(q) for q in x["q"]] if kind != "fa" else None
    ctx, new = _shape(case)
    seqs = [c + n for c, n in zip(ctx, new)]
    if kind == "decode":
        # the split count the vLLM shim plans for this batch, as an engine that calls the operator itself does
        s["seg"] = _segments(sum(new), hq)
        s["nsplit"] = pkg.vllm_shim.decode_splits(64, case["window"], hkv, len(seqs), "cuda", seqs, case["qlen"], hq)
    if kind in ("step", "mixed"):
        dec = sum(n for n in new[:case["seqs"]])
        s["seg"] = _segments(max(1, dec), hq)
        meta = pkg.vllm_shim.AttnMeta(x["qsl"], x["qsl_cpu"], x["lens"], x["bt"], max(seqs), True, *s["seg"],
                                      seq_lens_cpu=x["lens_cpu"])
        s["meta"] = meta
        s["layer"] = [pkg.vllm_shim.Gfx950Int8Attention(
            num_heads=hq, num_kv_heads=hkv, head_size=_DIM, scale=_SCALE, kv_quant_int8_per_token_head=True,
            is_rocm=True, is_decoder=True) for _ in s["caches"]]
        s["max_q"], s["tokens"] = max(new), sum(new)
    if kind == "step" and case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _step(s)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        s["replay"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["replay"]):
            _step(s)
    return s


def _unrouted(*a):
    raise RuntimeError("the batch was not routed to the operators")


def _route(s, i):
    c = s["caches"][i]
    if not s["layer"][i].route(s["q"][i], c.key_cache, c.value_cache, c.k_scale, c.v_scale, s["meta"], s["out"][i],
                               s["max_q"], s["tokens"], _unrouted):
        _unrouted()


def _step(s):
    write = s["pkg"].cache_write
    for i, c in enumerate(s["caches"]):
        new = s["new"][i]
        write(new[:, 0], new[:, 1], c.key_cache, c.value_cache, c.k_scale, c.v_scale, s["slots"])
        _route(s, i)


def run(state):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind == "step":
        if "replay" in s:
            s["replay"].replay()
        else:
            _step(s)
        return s["out"]
    if kind == "mixed":
        _route(s, 0)
        return s["out"]
    c = s["cache"] if kind == "write" else s["caches"][0]
    if kind == "write":
        s["pkg"].cache_write(s["key"], s["value"], c.key_cache, c.value_cache, c.k_scale, c.v_scale, s["slots"])
        return c.kv
    if kind == "decode":
        s["pkg"].decode(s["q"][0], c.key_cache, c.value_cache, c.k_scale, c.v_scale, s["bt"], s["lens"], s["qsl"],
                        s["out"][0], _SCALE, *s["seg"], case["seqs"], case["qlen"], s["nsplit"],
                        window=case["window"], causal=case["causal"])
        return s["out"]
    return [s["pkg"].forward_pth(s["q"][0], c.key_cache, c.value_cache, s["bt"], s["lens"], _SCALE, s["q_abs"],
                                 exact=case["exact"], max_keys=case["ctx"] + case["tokens"])]


def work(case):
    hq, hkv, kind = case["heads_q"], case["heads_kv"], case["kind"]
    if kind == "write":
        size = 4 if case["dtype"] == "fp32" else 2
        return {"bytes": case["tokens"] * (hkv * (2 * _DIM * size + _ROW) + 8), "flops": 0}
    ctx, new = _shape(case)
    layers, bs, window, causal = case.get("layers", 1), case["block_size"], case.get("window", -1), case.get("causal", True)
    keys = pairs = pages = 0
    for c, n in zip(ctx, new):
        lo = max(0, c - window + 1) if window > 0 else 0
        keys += c + n - lo
        pages += (c + n - 1) // bs - lo // bs + 1
        if window > 0:
            pairs += sum((p + 1 if causal else c + n) - max(0, p - window + 1) for p in range(c, c + n))
        else:
            pairs += n * c + n * (n + 1) // 2
    rows = sum(new) * hq
    qo = rows * _DIM * (8 if kind == "fa" else 4)
    b = keys * hkv * _ROW + qo + 4 * pages + 8 * len(ctx)
    if kind == "step":
        b += sum(new) * (hkv * 2 * _DIM * 2 + 8)  # the new tokens' K/V; their rows are counted with the keys
    return {"bytes": layers * b, "flops": layers * 4 * _DIM * hq * pairs}


def tolerance(case):
    if case["kind"] == "write":
        return "exact"
    if case["kind"] == "fa":
        if case["exact"]:
            return {"rel": 1e-5}  # 32-bit sums; measured 3e-7 to 1e-6
        # fp16 weights (measured 2.3e-4 to 4e-4), and over one long run of keys fp32 sums in which the 1152 of the
        # biased int8 widening is carried and cancelled at the end (measured 7.9e-3 at 63,488 keys, the 30-fold of
        # the weights' share; splits of a run shorten it)
        return {"rel": max(1.5e-3, 0.03 * min(1.0, ((case["ctx"] + case["tokens"]) / 63488) ** 1.5))}
    if case["kind"] == "mixed":
        return {"rel": 1.5e-3, "max": 0.02}  # fp16 outputs and weights; measured 3e-4 to 3.7e-4
    # fp16 outputs (measured 2.1e-4, the rounding alone); single values by some units in the last place
    return {"rel": 8e-4, "max": 4e-3}


def _attend(q, kv, bt, seq, first, window, causal):
    """q [n, hq, 256] float64 at positions first.., raw cache kv [pages, hkv, bs, 520]; float64 [n, hq, 256]."""
    n, hq, _ = q.shape
    hkv, bs = kv.shape[1], kv.shape[2]
    g = hq // hkv
    lo = max(0, first - window + 1) if window > 0 else 0
    pos = torch.arange(lo, seq, device="cuda")
    rows = kv[bt.long()[pos // bs], :, pos % bs]  # [keys, hkv, 520]
    out = torch.empty((n, hq, _DIM), dtype=torch.float64, device="cuda")
    step = max(1, min(n, (1 << 27) // max(1, g * pos.numel())))
    for h in range(hkv):
        r = rows[:, h].contiguous().view(-1, 2, 260)
        scales = r[:, :, _DIM:].contiguous().view(torch.float32).double()
        k, v = (r[:, j, :_DIM].double() * scales[:, j] for j in (0, 1))
        for i in range(0, n, step):
            m = min(step, n - i)
            p = torch.arange(first + i, first + i + m, device="cuda")
            see = torch.ones((m, pos.numel()), dtype=torch.bool, device="cuda")
            if causal:
                see &= pos[None, :] <= p[:, None]
            if window > 0:
                see &= p[:, None] - pos[None, :] < window
            x = q[i:i + m, h * g:(h + 1) * g].reshape(m * g, _DIM) @ k.t().contiguous() * _SCALE
            x.view(m, g, -1).masked_fill_(~see[:, None, :], -math.inf)
            out[i:i + m, h * g:(h + 1) * g] = (torch.softmax(x, -1) @ v).view(m, g, _DIM)
    return out


def exact(case, seed):
    if case["kind"] == "write":
        return None
    x = _inputs(case, seed)
    ctx, new = _shape(case)
    outs = []
    for i, kv in enumerate(x["kv"]):
        if case["kind"] == "step":  # store the new tokens' rows
            t = x["new"][i].float().cpu().transpose(1, 2)  # [T, hkv, 2, 256]
            s = t.abs().amax(-1, keepdim=True) / 127.0
            row = torch.cat([(t / s).round().clamp(-127, 127).to(torch.int8), s.view(torch.int8)], -1)
            bs = case["block_size"]
            kv[x["slots"] // bs, :, x["slots"] % bs] = row.reshape(t.shape[0], -1, _ROW).cuda()
        q = (x["q"][i][0].transpose(0, 1) if case["kind"] == "fa" else x["q"][i]).double()
        o, at = [], 0
        for b, (c, n) in enumerate(zip(ctx, new)):
            o.append(_attend(q[at:at + n], kv, x["bt"][b], c + n, c, case.get("window", -1), case.get("causal", True)))
            at += n
        o = torch.cat(o)
        outs.append(o.unsqueeze(0) if case["kind"] == "fa" else o)
    return outs
