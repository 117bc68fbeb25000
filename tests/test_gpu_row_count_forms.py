"""The forms a launch takes the query row counts in (``sas_attention_launch_lens``):
cumulative counts and uniform counts give bitwise what the arrays give, on every
kernel, with and without split items; rows of no batch come out zero; captured
calls share a zeroed counter array per capture and replay like eager calls."""

import ctypes

import pytest
import torch

from oracle import gen

pytestmark = pytest.mark.gpu

HAS_GPU = torch.cuda.is_available()
requires_gpu = pytest.mark.skipif(not HAS_GPU, reason="needs a ROCm GPU")

if HAS_GPU:
    from sparse_attn_sharedkv_amd import (_lib, api, sparse_attn_sharedkv,
                                          sparse_attn_sharedkv_metadata)


def _tnd(kw, rows, lead=0, tail=0):
    """The workload as TND: ``rows[b]`` query rows a sequence, ``lead`` and ``tail`` rows of none."""
    kw = dict(kw)
    n = lead + sum(rows) + tail
    h, d = kw["q"].shape[-2:]
    g = torch.Generator(device="cuda").manual_seed(n)
    kw["q"] = (torch.randn((n, h, d), generator=g, device="cuda") * 0.5).to(kw["q"].dtype)
    idx = kw.get("cmp_sparse_indices")
    if idx is not None:
        k = idx.shape[-1]
        kw["cmp_sparse_indices"] = torch.randint(0, 300, (n, 1, k), generator=g, device="cuda",
                                                 dtype=torch.int32)
    kw["cu_seqlens_q"] = torch.tensor([lead] + rows, dtype=torch.int32).cumsum(0).to(
        dtype=torch.int32, device="cuda")
    kw["layout_q"] = "TND"
    return kw


def _launch(prep, form, **fields):
    a = prep.args
    old = {f: getattr(a, f) for f in fields}
    for f, v in fields.items():
        setattr(a, f, v)
    a.phases = prep.phase_bits
    a.merge_sync = None
    prep.out.fill_(7.0)
    prep.lse.fill_(7.0)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = _lib.load().sas_attention_launch_lens(ctypes.byref(a), form, st)
    assert rc == _lib.SAS_OK, _lib.last_error()
    torch.cuda.synchronize()
    for f, v in old.items():
        setattr(a, f, v)
    return prep.out.clone(), prep.lse.clone()


# every kernel: one wave per SIMD (decode; several rows), row pairs, 128-head items, fp8 rows of
# 64- and 128-head items; lengths in lanes (up to 64 batches) and as scalar loads
FORMS = [
    ("swa_topk_decode_b32_h64_k512", 5, 0, 256), ("swa_topk_decode_b32_h64_k512", 70, 1, 256),
    ("swa_decode_b32_h64", 6, 3, 7), ("mla_decode_b64_h128_k2048", 3, 0, 64),
    ("mla_decode_b64_h128_k2048", 66, 1, 256), ("mla_fp8_decode_t128_h128_k2048", 3, 1, 256),
    ("mla_fp8_decode_t128_h128_k2048", 66, 0, 100), ("topk_decode_b2_h16_k256", 2, 2, 3),
]


@requires_gpu
@pytest.mark.parametrize("name,batch,more,cores", FORMS)
def test_forms_agree_and_unowned_rows_are_zero(name, batch, more, cores):
    print(f"[gpu-row-forms] {name} batch={batch} cores={cores}", flush=True)
    kw = gen.build_workload(name, device="cuda", seed=batch, batch=batch,
                            ctx_override=[900 + 7 * b for b in range(batch)])
    rows = [1 + (b * more) % 4 for b in range(batch)]
    for lead, tail in ((0, 0), (0, 5), (2, 1)):
        t = _tnd(kw, rows, lead, tail)
        prep = api.prepare(**t, schedule="host", core_num=cores)
        ref = _launch(prep, _lib.QLENS_ARRAYS)
        own = slice(lead, lead + sum(rows))
        got = _launch(prep, _lib.QLENS_CUMULATIVE, q_prefix=t["cu_seqlens_q"].data_ptr(),
                      act_q_lens=None)
        for r, o in zip(ref, got):
            assert torch.equal(r[own], o[own])
            assert not o[:lead].any() and not o[own.stop:].any()
        # the public call, scheduled on the host, on the GPU and from a schedule tensor
        for how in ("host", "device"):
            out, lse = sparse_attn_sharedkv(**t, schedule=how, core_num=cores,
                                            return_softmax_lse=True)
            assert torch.equal(out, got[0]) and torch.equal(lse, got[1]), how
    s = max(rows)
    b = dict(_tnd(kw, [s] * batch), layout_q="BSND", cu_seqlens_q=None)
    b["q"] = b["q"].view(batch, s, *b["q"].shape[1:])
    if b.get("cmp_sparse_indices") is not None:
        b["cmp_sparse_indices"] = b["cmp_sparse_indices"].view(batch, s, 1, -1)
    prep = api.prepare(**b, schedule="host", core_num=cores)
    ref = _launch(prep, _lib.QLENS_ARRAYS)
    got = _launch(prep, _lib.QLENS_UNIFORM, q_prefix=None, act_q_lens=None)
    assert torch.equal(ref[0], got[0]) and torch.equal(ref[1], got[1])


@requires_gpu
def test_schedule_of_fewer_batches_leaves_zero_rows():
    # a schedule tensor built for the first sequences only: the others' rows are zero
    kw = _tnd(gen.build_workload("swa_decode_b32_h64", device="cuda", seed=1, batch=6),
              [1, 2, 1, 3, 1, 2])
    md = sparse_attn_sharedkv_metadata(
        num_heads_q=64, num_heads_kv=1, head_dim=576, cu_seqlens_q=kw["cu_seqlens_q"][:4],
        seqused_kv=kw["seqused_kv"], layout_q="TND", has_cmp_kv=False, device="cuda")
    full = sparse_attn_sharedkv(**kw, schedule="device")
    out, lse = sparse_attn_sharedkv(**kw, metadata=md, return_softmax_lse=True)
    assert torch.equal(out[:4], full[:4]) and not out[4:].any() and not lse[4:].any()


def test_bad_forms_are_refused():
    lib = _lib_or_skip()
    a = _fields()
    assert lib.sas_attention_launch_lens(None, 0, None) == -1
    assert lib.sas_attention_launch_lens(ctypes.byref(a), 3, None) == -1
    a.q_prefix = None
    assert lib.sas_attention_launch_lens(ctypes.byref(a), 1, None) == -1
    a = _fields()
    a.act_q_lens = None
    assert lib.sas_attention_launch(ctypes.byref(a), None) == -1
    a.batch, a.total_tokens = 3, 4
    assert lib.sas_attention_launch_lens(ctypes.byref(a), 2, None) == -1


def _lib_or_skip():
    from sparse_attn_sharedkv_amd import _lib as binding
    return binding.load()


def _fields():
    from sparse_attn_sharedkv_amd import _lib as binding
    a = binding.SasAttnArgs()
    for f in ("q", "ori_kv", "ori_block_table", "q_prefix", "act_q_lens", "seqused_kv", "sinks",
              "metadata", "out", "lse"):
        setattr(a, f, 64)  # never read: every call here is refused first
    a.head_dim = 17
    return a


@requires_gpu
def test_captured_calls_share_counters_and_replay():
    # two graphs of two calls each (split items, merged in the kernel), replayed in
    # turn with eager calls between them: every replay is bitwise the eager call
    kws = [gen.build_workload("mla_decode_b64_h128_k2048", device="cuda", seed=s, batch=64)
           for s in (1, 2)]
    mds = [sparse_attn_sharedkv_metadata(
        num_heads_q=128, num_heads_kv=1, head_dim=576, seqused_kv=k["seqused_kv"], batch_size=64,
        max_seqlen_q=1, cmp_topk=2048, cmp_ratio=1, ori_win_left=-1, device="cuda") for k in kws]
    call = lambda i: sparse_attn_sharedkv(**kws[i], metadata=mds[i], return_softmax_lse=True)
    refs = [[x.clone() for x in call(i)] for i in range(2)]
    torch.cuda.synchronize()
    graphs, outs = [], []
    for g in range(2):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outs.append([call(i) for i in range(2)])
        graphs.append(graph)
    for r in range(6):
        graphs[r % 2].replay()
        eager = call(r % 2)
        torch.cuda.synchronize()
        for i in range(2):
            assert all(torch.equal(x, y) for x, y in zip(outs[r % 2][i], refs[i])), r
        assert all(torch.equal(x, y) for x, y in zip(eager, refs[r % 2]))
