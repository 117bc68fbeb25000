"""The work whose speed is tracked: attention and cache-writer calls as serving programs make them.

Every case goes through the package's public entry points. Attention cases differ in how the
program calls them (``how``):

* ``graph``  a decode step captured once in a HIP graph and replayed, its schedule built on the
             GPU beforehand and shared by a model's layers (the way a serving loop decodes);
* ``eager``  one call with a schedule tensor built on the GPU beforehand (eager decode);
* ``device`` one call that builds its schedule on the GPU (``schedule="device"``);
* ``step``   schedule and call together, both on the GPU: a step whose lengths are new;
* ``flash``  one ``sparse_flash_mla`` call, which schedules on the host (prefill).

Queries and cache rows are N(0, 1), so scaled scores have a standard deviation of about 1 and a
row's softmax weights span the three decades that trained heads show; top-k ids are a uniform
subset of the causal prefix in random order; block tables scatter every sequence over the pool.
"""

import math

import torch

from sparse_attn_sharedkv_amd import (append_kv_fp8, sparse_attn_sharedkv,
                                      sparse_attn_sharedkv_metadata, sparse_flash_mla)

FP8_ROW = 656          # 512 e4m3 + 4 fp32 block scales + 64 bf16
D_V = 512
EXACT_FLOPS = 0.4e12   # a 64-bit reference over this takes too long

_ATTN = dict(kind="attn", how="graph", batch=1, q_lo=1, q_hi=1, heads=64, d=576, window=-1,
             ratio=1, topk=0, ctx_lo=1024, ctx_hi=1024, block=64, layout="BSND", dtype="bf16",
             kv="native", fp8_qk=False)


def _attn(**over):
    return dict(_ATTN, **over)


def listed():
    return [
        # the smallest call: two short sequences with few heads (a test or a draft model's step)
        _attn(name="topk_decode_b2_h16", how="eager", batch=2, heads=16, topk=256),
        # sliding-window layers of a decode batch with ragged contexts
        _attn(name="swa_decode_b32_h64", batch=32, window=127, ctx_lo=2048, ctx_hi=8192),
        # window + top-k of the compressed cache, a decode batch at one context
        _attn(name="swa_topk_decode_b32_h64", batch=32, window=127, ratio=4, topk=512,
              ctx_lo=16384, ctx_hi=16384),
        # sparse MLA decode of a full batch: every head over the top 2048 rows
        _attn(name="mla_decode_b64_h128", batch=64, heads=128, topk=2048, ctx_lo=32768,
              ctx_hi=32768),
        # the same with a speculative second row, one eager call that schedules on the GPU
        _attn(name="mla_mtp_decode_b64_h128", how="device", batch=64, q_lo=2, q_hi=2, heads=128,
              topk=2048, ctx_lo=32768, ctx_hi=32768),
        # long-context sparse MLA over an fp8 cache, ragged
        _attn(name="mla_fp8_decode_b128_h128", batch=128, heads=128, topk=2048, ctx_lo=32768,
              ctx_hi=131072, layout="TND", kv="fp8"),
        # a smaller fp8 batch with fp8 query products, contexts shorter than the top-k among them
        _attn(name="mla_fp8qk_decode_b13_h128", batch=13, heads=128, topk=2048, ctx_lo=700,
              ctx_hi=20000, layout="TND", kv="fp8", fp8_qk=True),
        # a mixed step: decode rows and prefill chunks of odd lengths in one ragged call
        _attn(name="mixed_step_b23_h64_fp16", how="step", batch=23, q_lo=1, q_hi=157, d=512,
              window=127, ratio=4, topk=512, ctx_lo=300, ctx_hi=6000, layout="TND", dtype="fp16"),
        # 8K prefill: window only; window and every compressed row; window and top-k
        _attn(name="swa_prefill_t8192_h64", how="flash", q_lo=8192, q_hi=8192, d=512, window=127,
              ctx_lo=8192, ctx_hi=8192, block=128, layout="TND"),
        _attn(name="cfa_prefill_t8192_h64", how="flash", q_lo=8192, q_hi=8192, d=512, window=127,
              ratio=128, topk=-1, ctx_lo=8192, ctx_hi=8192, block=128, layout="TND"),
        _attn(name="scfa_prefill_t8192_h64", how="flash", q_lo=8192, q_hi=8192, d=512, window=127,
              ratio=4, topk=512, ctx_lo=8192, ctx_hi=8192, block=128, layout="TND"),
        # the fp8 cache writer on a prefill's rows
        dict(name="append_fp8_n16384", kind="append", n=16384, pool=65536),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["topk", "topk", "window", "window", "fp8", "fp8", "prefill", "prefill",
                       "mixed", "append"])
    if kind == "append":
        n = _log_int(rng, 1, 65536)
        return dict(kind="append", n=n, pool=n + rng.randrange(1, 65536))
    how = rng.choice(["graph", "graph", "eager", "device", "step"])
    layout = rng.choice(["BSND", "TND"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    ctx_hi = _log_int(rng, 600, 32768)
    ctx_lo = rng.choice([ctx_hi, rng.randrange(ctx_hi // 4, ctx_hi + 1)])
    block = rng.choice([16, 64, 64, 128])
    c = _attn(how=how, layout=layout, dtype=dtype, ctx_lo=ctx_lo, ctx_hi=ctx_hi, block=block,
              batch=_log_int(rng, 1, 128), q_lo=1, q_hi=1)
    if kind == "topk":
        rows = rng.choice([1, 1, 1, 2, 3])
        c.update(heads=rng.choice([16, 32, 64, 96, 128, 128]), q_lo=rows, q_hi=rows,
                 topk=rng.choice([256, 512, 1024, 2048, 2048, rng.randrange(100, 2049)]))
    elif kind == "window":
        c.update(heads=rng.choice([16, 32, 48, 64, 64, 128]), d=rng.choice([512, 576]),
                 window=rng.choice([63, 127, 127, 511]))
        sel = rng.choice(["none", "dense", "topk"])
        if sel == "dense":
            c.update(ratio=128, topk=-1)
        elif sel == "topk":
            c.update(ratio=4, topk=rng.choice([256, 512, rng.randrange(50, 1025)]))
    elif kind == "fp8":
        c.update(kv="fp8", dtype="bf16", heads=rng.choice([64, 128, 128]), topk=2048,
                 fp8_qk=rng.choice([False, True]))
    elif kind == "prefill":
        t = _log_int(rng, 200, 8192)
        c.update(how=rng.choice(["flash", "device"]), layout="TND", batch=rng.choice([1, 1, 2, 3]),
                 d=rng.choice([512, 576]), heads=64, window=127)
        c["ctx_hi"] = t + rng.choice([0, 0, rng.randrange(0, 4097)])
        c["ctx_lo"] = c["ctx_hi"]
        c["q_hi"] = max(t // c["batch"], 1)
        c["q_lo"] = rng.choice([c["q_hi"], max(c["q_hi"] // 2, 1)])
        sel = rng.choice(["none", "dense", "topk"])
        if sel == "dense":
            c.update(ratio=128, topk=-1)
        elif sel == "topk":
            c.update(ratio=4, topk=512)
        if rng.random() < 0.3:
            c.update(heads=128, q_lo=(c["q_lo"] + 3) // 4, q_hi=(c["q_hi"] + 3) // 4)
    else:
        c.update(how=rng.choice(["device", "step"]), layout="TND", batch=rng.randrange(5, 41),
                 q_hi=rng.randrange(20, 161), d=512, window=127, ctx_lo=200)
        c["ctx_hi"] = max(c["ctx_hi"], 600)
        if rng.random() < 0.6:
            c.update(ratio=4, topk=512)
    return c


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _lengths(case, seed):
    """Per-sequence query rows and context lengths (never shorter than the rows). The row counts
    are the case's own, in an order of the seed's, so every seed has as many tokens."""
    b, lo, hi = case["batch"], case["q_lo"], case["q_hi"]
    g = torch.Generator().manual_seed(seed * 8 + 1)
    if case["layout"] == "BSND" or lo == hi:
        rows = torch.full((b,), hi)
    else:
        own = torch.Generator().manual_seed(lo + 1000 * hi + b)
        rows = torch.randint(lo, hi + 1, (b,), generator=own)
        if lo == 1:  # a mixed step: most sequences decode one row
            rows = torch.where(torch.rand(b, generator=own) < 0.7, torch.ones_like(rows), rows)
        rows = rows[torch.randperm(b, generator=g)]
    kv = torch.randint(case["ctx_lo"], case["ctx_hi"] + 1, (b,), generator=g)
    return rows.tolist(), torch.maximum(kv, rows).tolist()


def _table(lens, block, g):
    """A pool's block table: every sequence's blocks are a random slice of the pool."""
    per = [max((n + block - 1) // block, 1) for n in lens]
    perm = torch.randperm(sum(per), generator=g, device="cuda").to(torch.int32)
    table = torch.full((len(lens), max(per)), -1, dtype=torch.int32, device="cuda")
    at = 0
    for i, n in enumerate(per):
        table[i, :n] = perm[at:at + n]
        at += n
    return sum(per), table


def _fp8_rows(x):
    """bf16 rows [n, 576] as 656-byte rows: e4m3 of x * 448 / amax per 128 dims, scales, rope."""
    n = x.shape[0]
    lat = x[:, :512].float().reshape(n, 4, 128)
    scale = lat.abs().amax(dim=2) / 448.0
    scale = torch.where(scale > 0, scale, torch.ones_like(scale))
    e4 = (lat / scale[:, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn).reshape(n, 512)
    return torch.cat([e4.view(torch.uint8), scale.view(torch.uint8),
                      x[:, 512:].contiguous().view(torch.uint8)], dim=1)


def _from_fp8_rows(rows):
    """What the attention reads from 656-byte rows: bf16(e4m3 * scale) and the rope dims."""
    n = rows.shape[0]
    lat = rows[:, :512].contiguous().view(torch.float8_e4m3fn).float().reshape(n, 4, 128)
    scale = rows[:, 512:528].contiguous().view(torch.float32)
    lat = (lat * scale[:, :, None]).to(torch.bfloat16).reshape(n, 512)
    return torch.cat([lat, rows[:, 528:].contiguous().view(torch.bfloat16)], dim=1)


def _pool(case, lens, g, dtype):
    blocks, table = _table(lens, case["block"], g)
    n, d = blocks * case["block"], case["d"]
    width, kind = (FP8_ROW, torch.uint8) if case["kv"] == "fp8" else (d, dtype)
    pool = torch.empty((n, width), dtype=kind, device="cuda")
    for at in range(0, n, 1 << 20):
        x = torch.randn((min(1 << 20, n - at), d), generator=g, device="cuda",
                        dtype=torch.bfloat16 if case["kv"] == "fp8" else dtype)
        pool[at:at + x.shape[0]] = _fp8_rows(x) if case["kv"] == "fp8" else x
    return pool.view(blocks, case["block"], 1, width), table


def _topk(case, rows, lens, g):
    """[tokens, K] int32: a random K-subset of each row's causal prefix, -1 padded."""
    k = case["topk"]
    thr = torch.cat([(torch.arange(n - r, n, device="cuda") + 1) // case["ratio"]
                     for r, n in zip(rows, lens)])
    out = torch.full((thr.numel(), k), -1, dtype=torch.int32, device="cuda")
    widest = max(int(thr.max()), 1)
    step = max((1 << 27) // widest, 1)
    for at in range(0, thr.numel(), step):
        t = thr[at:at + step, None]
        keys = torch.rand((t.shape[0], widest), generator=g, device="cuda")
        keys.masked_fill_(torch.arange(widest, device="cuda") >= t, 2.0)
        top = keys.topk(min(k, widest), dim=1, largest=False)
        idx = torch.where(top.values < 2.0, top.indices, -1).to(torch.int32)
        out[at:at + t.shape[0], :idx.shape[1]] = idx
    return out


def _inputs(case, seed):
    dtype = torch.float16 if case["dtype"] == "fp16" else torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(seed)
    rows, lens = _lengths(case, seed)
    t, h, d = sum(rows), case["heads"], case["d"]
    q = torch.randn((t, h, d), generator=g, device="cuda", dtype=dtype)
    ori, ori_bt = _pool(case, lens, g, dtype)
    args = dict(ori_kv=ori, ori_block_table=ori_bt, softmax_scale=1.0 / math.sqrt(d),
                cmp_ratio=case["ratio"], ori_win_left=case["window"], layout_q=case["layout"],
                head_dim_v=D_V, return_softmax_lse=True,
                seqused_kv=torch.tensor(lens, dtype=torch.int32, device="cuda"))
    if case["topk"]:
        if case["window"] < 0:  # pure top-k: the raw cache is what the ids select from
            args.update(cmp_kv=ori, cmp_block_table=ori_bt)
        else:
            pool, table = _pool(case, [max(n // case["ratio"], 1) for n in lens], g, dtype)
            args.update(cmp_kv=pool, cmp_block_table=table)
    if case["window"] < 0:
        args["sinks"] = torch.full((h,), float("-inf"), device="cuda")
    else:
        args["sinks"] = torch.rand((h,), generator=g, device="cuda") * 2 - 1
    idx = _topk(case, rows, lens, g) if case["topk"] > 0 else None
    if case["layout"] == "TND":
        cu = torch.tensor([0] + rows, dtype=torch.int32).cumsum(0).to(torch.int32)
        args.update(q=q, cu_seqlens_q=cu.cuda(),
                    cmp_sparse_indices=None if idx is None else idx.unsqueeze(1))
    else:
        s = rows[0]
        args.update(q=q.view(-1, s, h, d), cmp_sparse_indices=None if idx is None else
                    idx.view(-1, s, 1, idx.shape[1]))
    if case["kv"] == "fp8":
        args.update(kv_cache_dtype="fp8_ds_mla", fp8_qk=case["fp8_qk"])
    return args, rows, lens


def _metadata(case, args):
    tnd = case["layout"] == "TND"
    return sparse_attn_sharedkv_metadata(
        num_heads_q=case["heads"], num_heads_kv=1, head_dim=case["d"],
        cu_seqlens_q=args["cu_seqlens_q"] if tnd else None, seqused_kv=args["seqused_kv"],
        batch_size=case["batch"], max_seqlen_q=case["q_hi"], max_seqlen_kv=case["ctx_hi"],
        cmp_topk=max(case["topk"], 0), cmp_ratio=case["ratio"], ori_win_left=case["window"],
        layout_q=case["layout"], has_cmp_kv=case["topk"] != 0, device="cuda",
        kv_cache_dtype=args.get("kv_cache_dtype"), fp8_qk=case["fp8_qk"])


def _append_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rows = torch.randn((case["n"], 576), generator=g, device="cuda", dtype=torch.bfloat16)
    slots = torch.randperm(case["pool"], generator=g, device="cuda")[:case["n"]].to(torch.int32)
    return rows, slots


def prepare(case, seed):
    if case["kind"] == "append":
        rows, slots = _append_inputs(case, seed)
        cache = torch.zeros((case["pool"], 1, 1, FP8_ROW), dtype=torch.uint8, device="cuda")
        return dict(kind="append", cache=cache, rows=rows, slots=slots)
    args, _, _ = _inputs(case, seed)
    how = case["how"]
    state = dict(kind=how, case=case, args=args)
    if how in ("graph", "eager"):
        args["metadata"] = _metadata(case, args)
    elif how == "device":
        args["schedule"] = "device"
    if how == "graph":
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):  # first use outside the capture
            sparse_attn_sharedkv(**args)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            state["out"] = sparse_attn_sharedkv(**args)
        state["graph"] = graph
    return state


def run(state):
    kind = state["kind"]
    if kind == "append":
        append_kv_fp8(state["cache"], state["rows"], state["slots"])
        return state["cache"]
    if kind == "graph":
        state["graph"].replay()
        return state["out"]
    if kind == "flash":
        return sparse_flash_mla(**state["args"])
    if kind == "step":
        return sparse_attn_sharedkv(metadata=_metadata(state["case"], state["args"]),
                                    **state["args"])
    return sparse_attn_sharedkv(**state["args"])


# ---------------------------------------------------------------------------
# What a pass cannot do without, how close results must be, and the 64-bit answer
# ---------------------------------------------------------------------------

def work(case):
    """Every input read once, every output written once; 2 (d_qk + d_v) flops per head and row."""
    if case["kind"] == "append":
        return dict(bytes=case["n"] * (2 * 576 + 4 + FP8_ROW), flops=0)
    rows, lens = _lengths(case, 1)  # (the counts of one seed: others differ by little)
    ratio, k, win = case["ratio"], case["topk"], case["window"]
    attended = distinct = 0
    for r, n in zip(rows, lens):
        first = n - r
        for s in range(first, n):
            attended += s + 1 - max(s - win, 0) if win >= 0 else 0
            attended += 0 if k == 0 else (s + 1) // ratio if k < 0 else min((s + 1) // ratio, k)
        distinct += n - max(first - win, 0) if win >= 0 else 0
        if k:
            top = n // ratio
            distinct += top if k < 0 else min(top, k * r)
    t, h, d = sum(rows), case["heads"], case["d"]
    row_bytes = FP8_ROW if case["kv"] == "fp8" else 2 * d
    nbytes = distinct * (row_bytes + 4) + t * h * (2 * d + 2 * D_V + 4) + t * max(k, 0) * 4
    return dict(bytes=nbytes, flops=2 * attended * h * (d + D_V))


def tolerance(case):
    """About four times what the results are off the 64-bit answer, which their type's rounding
    of weights and outputs gives (2e-3 in bf16, 2.6e-4 in fp16). With fp8 queries the answer is
    off by what the queries lost, which any implementation of that form shares."""
    if case["kind"] == "append":
        return "exact"
    return dict(rel=1e-3) if case["dtype"] == "fp16" else dict(rel=8e-3)


def exact(case, seed):
    if case["kind"] == "append" or work(case)["flops"] > EXACT_FLOPS:
        return None
    args, rows, lens = _inputs(case, seed)
    h, d = case["heads"], case["d"]
    q = args["q"].reshape(-1, h, d)
    idx = args["cmp_sparse_indices"]
    idx = None if idx is None else idx.reshape(q.shape[0], -1)
    out = torch.zeros((q.shape[0], h, D_V), dtype=torch.float64, device="cuda")
    lse = torch.zeros((q.shape[0], h), dtype=torch.float64, device="cuda")
    sink = args["sinks"].double()

    def rows_of(pool, table, pos):
        at = table[pos // case["block"]].long() * case["block"] + pos % case["block"]
        got = pool.reshape(-1, pool.shape[-1])[at.reshape(-1)]
        got = _from_fp8_rows(got) if case["kv"] == "fp8" else got
        return got.double().view(*pos.shape, d)

    tok = 0
    for b, (r, n) in enumerate(zip(rows, lens)):
        for s0 in range(n - r, n, 64):
            pos = torch.arange(s0, min(s0 + 64, n), device="cuda")[:, None]
            kv, ok = [], []
            if case["window"] >= 0:
                p = pos - case["window"] + torch.arange(case["window"] + 1, device="cuda")
                kv.append(rows_of(args["ori_kv"], args["ori_block_table"][b], p.clamp(min=0)))
                ok.append(p >= 0)
            if case["topk"]:
                thr = (pos + 1) // case["ratio"]
                if idx is None:
                    p = torch.arange(int(thr.max()), device="cuda").expand(pos.shape[0], -1)
                else:
                    p = idx[tok:tok + pos.shape[0]].long()
                kv.append(rows_of(args["cmp_kv"], args["cmp_block_table"][b], p.clamp(min=0)))
                ok.append((p >= 0) & (p < thr))
            kv, ok = torch.cat(kv, 1), torch.cat(ok, 1)
            x = torch.bmm(kv, q[tok:tok + pos.shape[0]].double().transpose(1, 2).contiguous())
            x = (x * args["softmax_scale"]).masked_fill(~ok[:, :, None], float("-inf"))
            x = x.transpose(1, 2).contiguous()  # [rows, heads, positions]
            l = torch.logaddexp(torch.logsumexp(x, 2), sink)
            w = torch.exp(x - l[:, :, None])
            out[tok:tok + pos.shape[0]] = torch.bmm(w, kv[:, :, :D_V].contiguous())
            lse[tok:tok + pos.shape[0]] = l
            tok += pos.shape[0]
    shape = args["q"].shape[:-2]
    return out.view(*shape, h, D_V), lse.view(*shape, h)
