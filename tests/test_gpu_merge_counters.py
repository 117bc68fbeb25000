"""Arrival counters of the in-kernel merge when a call's lengths are not its schedule's.

A schedule (a ``metadata`` tensor built once per batch shape, a captured call) may run
with lists that have become shorter or longer than it was made for, down to empty ones
whose later pieces hold nothing. Each such call gives bitwise what the separate merge
kernel gives, and leaves the counters at zero: the calls after it, of other lengths or
of the scheduled ones again, are not touched by it. Eager calls, replays of a graph,
and two graphs replayed at once on two streams.
"""

import pytest
import torch

from oracle import gen

pytestmark = pytest.mark.gpu

HAS_GPU = torch.cuda.is_available()
requires_gpu = pytest.mark.skipif(not HAS_GPU, reason="needs a ROCm GPU")

if HAS_GPU:
    from sparse_attn_sharedkv_amd import api

# every kernel that merges: one wave per SIMD (32- and 64-head items, one and several rows),
# row pairs, 128-head items of native and fp8 rows; items of 2 to 16 pieces
CASES = [
    ("h16", 4, 24, None, 1, 4000), ("mla_decode_b64_h128_k2048", 8, 100, 64, 1, 3000),
    ("mla_decode_b64_h128_k2048", 8, 256, 128, 1, 3000), ("mla_decode_b64_h128_k2048", 5, 7, 128, 1, 3000),
    ("mla_fp8_decode_t128_h128_k2048", 6, 64, 128, 1, 3000),
    ("swa_topk_decode_b32_h64_k512", 5, 24, None, 1, 4000),
    ("swa_topk_decode_b32_h64_k512", 4, 64, None, 3, 4000), ("dense", 4, 64, None, 3, 4000),
]
# lists of a few and of many blocks of 64 positions, at and beside their edges; empty ones
LENGTHS = [0, 1, 63, 64, 65, 127, 128, 129, 192, 320, 640, 961, 1024, 1025, 1999, 2048, 3500]


def _workload(name, batch, rows, full, seed):
    kw = gen.build_workload("swa_topk_decode_b32_h64_k512" if name in ("dense", "h16") else name,
                            device="cuda", seed=seed, batch=batch, ctx_override=[full] * batch)
    if name == "dense":
        kw["cmp_sparse_indices"] = kw["topk_cmp"] = None
    elif name == "h16":
        kw["q"], kw["sinks"] = kw["q"][..., :16, :], kw["sinks"][:16].contiguous()
    g = torch.Generator(device="cuda").manual_seed(seed)
    h, d = kw["q"].shape[-2:]
    kw["q"] = (torch.randn((batch * rows, h, d), generator=g, device="cuda") * 0.5).to(kw["q"].dtype)
    if kw.get("cmp_sparse_indices") is not None:
        k = kw["cmp_sparse_indices"].shape[-1]
        kw["cmp_sparse_indices"] = torch.randint(0, full // 5, (batch * rows, 1, k), generator=g,
                                                 device="cuda", dtype=torch.int32)
    kw["cu_seqlens_q"] = torch.arange(batch + 1, dtype=torch.int32, device="cuda") * rows
    kw["layout_q"] = "TND"
    # room for longer lists than the scheduled ones
    kw["ori_block_table"] = kw["ori_block_table"].clamp(min=0).repeat(1, 2)
    if kw.get("cmp_block_table") is not None:
        kw["cmp_block_table"] = kw["cmp_block_table"].clamp(min=0).repeat(1, 2)
    return kw


def _prepare(kw, cores, m_base, separate):
    # (_stream_schedule: the launch reads cu_seqlens_q and seqused_kv where they are)
    prep = api.prepare(**kw, core_num=cores, _m_base=m_base, _separate_merge=separate,
                       _stream_schedule=True)
    assert prep.args.num_fd > 0, "nothing is split"
    assert prep.args.seqused_kv == kw["seqused_kv"].data_ptr()
    return prep


def _launch(prep):
    prep.out.fill_(float("nan"))
    prep.lse.fill_(float("nan"))
    api.launch(prep)
    return prep.out, prep.lse


def _same(got, ref, what):
    for a, b in zip(got, ref):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), what


@requires_gpu
@pytest.mark.parametrize("name,batch,cores,m_base,rows,full", CASES)
def test_calls_of_other_lengths_leave_no_trace(name, batch, cores, m_base, rows, full):
    print(f"[gpu-merge-counters] {name} batch={batch} cores={cores} rows={rows}", flush=True)
    kw = _workload(name, batch, rows, full, seed=cores)
    lens = kw["seqused_kv"]
    sep, prep, cap = (_prepare(kw, cores, m_base, s) for s in (True, False, False))
    scheduled = [x.clone() for x in _launch(sep)]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        api.launch(cap)
    for i, base in enumerate(LENGTHS):
        lens.copy_(torch.tensor([LENGTHS[(i + 5 * b) % len(LENGTHS)] if b % 2 else base
                                 for b in range(batch)], dtype=torch.int32))
        ref = [x.clone() for x in _launch(sep)]
        _same(_launch(prep), ref, ("eager", base))
        cap.out.fill_(float("nan"))
        graph.replay()
        _same((cap.out, cap.lse), ref, ("replay", base))
        lens.fill_(full)  # the scheduled lengths again, right behind
        _same(_launch(prep), scheduled, ("eager after", base))
        cap.out.fill_(float("nan"))
        graph.replay()
        _same((cap.out, cap.lse), scheduled, ("replay after", base))
    torch.cuda.synchronize()
    for buf in api._MERGE_SYNC.values():
        assert not buf.any(), "arrival counters left nonzero"


@requires_gpu
@pytest.mark.parametrize("name,batch,cores,m_base,rows,full",
                         [c for c in CASES if c[4] > 1] + [CASES[2]])
def test_calls_of_fewer_rows_leave_no_trace(name, batch, cores, m_base, rows, full):
    # split items whose query rows are gone: what such a call gives for the others is
    # not defined, the calls after it are as ever
    print(f"[gpu-merge-counters] rows: {name} batch={batch} cores={cores} rows={rows}", flush=True)
    kw = _workload(name, batch, rows, full, seed=cores)
    cu, was = kw["cu_seqlens_q"], kw["cu_seqlens_q"].clone()
    sep, prep, cap = (_prepare(kw, cores, m_base, s) for s in (True, False, False))
    scheduled = [x.clone() for x in _launch(sep)]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        api.launch(cap)
    for counts in ([0] * batch, [rows - 1] * batch, [rows * (b % 2) for b in range(batch)],
                   [rows * (b == 0) for b in range(batch)]):
        cu.copy_(torch.tensor([0] + counts).cumsum(0).to(torch.int32))
        _launch(prep)
        graph.replay()
        cu.copy_(was)
        _same(_launch(prep), scheduled, ("eager after", counts))
        cap.out.fill_(float("nan"))
        graph.replay()
        _same((cap.out, cap.lse), scheduled, ("replay after", counts))
    torch.cuda.synchronize()
    for buf in api._MERGE_SYNC.values():
        assert not buf.any(), "arrival counters left nonzero"


@requires_gpu
def test_two_graphs_at_once_on_two_streams():
    kws = [_workload("mla_decode_b64_h128_k2048", 8, 1, 3000, seed=s) for s in (1, 2)]
    refs, preps, graphs = [], [], []
    for kw in kws:
        refs.append([x.clone() for x in _launch(_prepare(kw, 64, 128, True))])
        preps.append(_prepare(kw, 64, 128, False))
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1]):
            for _ in range(8):
                api.launch(preps[-1])
    assert preps[0].args.merge_sync != preps[1].args.merge_sync
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    for r in range(5):
        for p in preps:
            p.out.fill_(float("nan"))
        torch.cuda.synchronize()
        for g, st in zip(graphs, streams):
            with torch.cuda.stream(st):
                g.replay()
        torch.cuda.synchronize()
        for p, ref in zip(preps, refs):
            _same((p.out, p.lse), ref, r)
