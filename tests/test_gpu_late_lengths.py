"""Host-scheduled calls read their lengths back behind the rest of the preparation and
keep their schedules on the GPU: bitwise the results of a call staged step by step, for
lengths changed in place, more length sets than are kept, and several streams."""

import pytest
import torch

from oracle import gen

pytestmark = pytest.mark.gpu

HAS_GPU = torch.cuda.is_available()
requires_gpu = pytest.mark.skipif(not HAS_GPU, reason="needs a ROCm GPU")

if HAS_GPU:
    from sparse_attn_sharedkv_amd import api, sparse_attn_sharedkv


def _staged(kw):
    """The call with its lengths read before anything else, its schedule copied for it."""
    prep = api.prepare(**kw)
    api.launch(prep)
    return api.finalize(prep, True)


def _same(kw, what):
    ref = _staged(kw)
    got = sparse_attn_sharedkv(**kw, return_softmax_lse=True)
    for a, b in zip(got, ref):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), what


def _workload(layout, batch=5):
    kw = gen.build_workload("swa_topk_decode_b32_h64_k512", device="cuda", seed=3, batch=batch,
                            ctx_override=[900 + 7 * b for b in range(batch)])
    if layout == "TND":
        q = kw["q"]
        kw["q"] = q.reshape(-1, *q.shape[-2:]).contiguous()
        idx = kw["cmp_sparse_indices"]
        kw["cmp_sparse_indices"] = idx.reshape(-1, *idx.shape[-2:])
        kw["cu_seqlens_q"] = torch.arange(batch + 1, dtype=torch.int32, device="cuda")
        kw["layout_q"] = "TND"
    return kw


@requires_gpu
@pytest.mark.parametrize("layout", ["TND", "BSND"])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_lengths_changed_in_place(layout, dtype):
    kw = _workload(layout)
    kw["seqused_kv"] = kw["seqused_kv"].to(dtype)
    for n in (900, 1, 0, 129, 640, 900):
        kw["seqused_kv"].copy_(torch.arange(5).cuda() * 3 + n)
        _same(kw, (layout, n))
    if layout == "TND":
        for rows in ([1, 0, 2, 1, 1], [0, 0, 0, 0, 5], [0, 1, 1, 0, 1]):
            kw["cu_seqlens_q"].copy_(torch.tensor([0] + rows).cumsum(0))
            _same(kw, rows)


@requires_gpu
def test_more_length_sets_than_are_kept_on_several_streams():
    kw = _workload("TND")
    streams = [torch.cuda.current_stream(), torch.cuda.Stream(), torch.cuda.Stream()]
    sets = [300 + 5 * i for i in range(api._GPU_SCHEDULES_MAX + 3)] + [300, 305, 310]
    refs = []
    for n in sets:
        kw["seqused_kv"] = torch.arange(n, n + 5, dtype=torch.int32, device="cuda")
        refs.append((kw["seqused_kv"], _staged(kw)))
    torch.cuda.synchronize()
    outs = []
    for i, (lens, _) in enumerate(refs):
        kw["seqused_kv"] = lens
        with torch.cuda.stream(streams[i % 3]):
            outs.append(sparse_attn_sharedkv(**kw, return_softmax_lse=True))
    torch.cuda.synchronize()
    assert len(api._GPU_SCHEDULES) <= api._GPU_SCHEDULES_MAX
    for got, (lens, ref) in zip(outs, refs):
        for a, b in zip(got, ref):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), lens


@requires_gpu
def test_what_the_host_scheduler_refuses_stays_refused():
    kw = _workload("TND")
    kw["seqused_kv"][2] = -1
    with pytest.raises(Exception) as early:
        _staged(kw)
    with pytest.raises(type(early.value)) as late:
        sparse_attn_sharedkv(**kw)
    assert str(late.value) == str(early.value)
