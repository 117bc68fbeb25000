"""Launches with cumulative row counts zero exactly the rows of no batch: for more FA rows
than the schedule uses (rows out of use behind, between and before the others), and where
no sequence has a query row at all."""

import ctypes

import pytest
import torch

from oracle import gen

pytestmark = pytest.mark.gpu

HAS_GPU = torch.cuda.is_available()
requires_gpu = pytest.mark.skipif(not HAS_GPU, reason="needs a ROCm GPU")

if HAS_GPU:
    from sparse_attn_sharedkv_amd import _lib, api, sparse_attn_sharedkv
    from sparse_attn_sharedkv_amd.metadata import SAS_META_SIZE


def _tnd(name, batch, rows, lead, tail):
    kw = gen.build_workload(name, device="cuda", seed=batch, batch=batch,
                            ctx_override=[900 + 7 * b for b in range(batch)])
    n = lead + sum(rows) + tail
    h, d = kw["q"].shape[-2:]
    g = torch.Generator(device="cuda").manual_seed(n)
    kw["q"] = (torch.randn((n, h, d), generator=g, device="cuda") * 0.5).to(kw["q"].dtype)
    if kw.get("cmp_sparse_indices") is not None:
        k = kw["cmp_sparse_indices"].shape[-1]
        kw["cmp_sparse_indices"] = torch.randint(0, 200, (n, 1, k), generator=g, device="cuda",
                                                 dtype=torch.int32)
    kw["cu_seqlens_q"] = torch.tensor([lead] + rows).cumsum(0).to(torch.int32).cuda()
    kw["layout_q"] = "TND"
    return kw


def _launch(prep, cu, md, num_fa):
    a = prep.args
    a.q_prefix, a.act_q_lens, a.merge_sync = cu.data_ptr(), None, None
    a.metadata, a.num_fa, a.phases = md.data_ptr(), num_fa, prep.phase_bits
    prep.out.fill_(7.0)
    prep.lse.fill_(7.0)
    rc = _lib.load().sas_attention_launch_lens(
        ctypes.byref(a), _lib.QLENS_CUMULATIVE,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == _lib.SAS_OK, _lib.last_error()
    torch.cuda.synchronize()
    return prep.out.clone(), prep.lse.clone()


@requires_gpu
@pytest.mark.parametrize("name,batch,more,cores", [
    ("topk_decode_b2_h16_k256", 2, 2, 3), ("swa_topk_decode_b32_h64_k512", 5, 0, 40),
    ("swa_decode_b32_h64", 6, 3, 7), ("mla_decode_b64_h128_k2048", 66, 1, 100),
    ("mla_fp8_decode_t128_h128_k2048", 3, 1, 64), ("mla_fp8_decode_t128_h128_k2048", 40, 0, 30),
])
def test_rows_out_of_use(name, batch, more, cores):
    print(f"[gpu-rows-out-of-use] {name} batch={batch} cores={cores}", flush=True)
    rows = [1 + (b * more) % 4 for b in range(batch)]
    t = _tnd(name, batch, rows, 2, 11)
    prep = api.prepare(**t, schedule="host", core_num=cores)
    md = next(x for x in prep.keep if x is not None and x.numel() == SAS_META_SIZE)
    used, cu = prep.args.num_fa, t["cu_seqlens_q"]
    ref = _launch(prep, cu, md, used)
    own = slice(2, 2 + sum(rows))
    assert not ref[0][:2].any() and not ref[0][own.stop:].any() and not ref[1][own.stop:].any()
    assert (ref[0][own] != 7.0).any()
    fa = md[:used * _lib.FA_METADATA_SIZE].view(used, _lib.FA_METADATA_SIZE)
    off = torch.zeros_like(fa[:1])
    spread = [off, off]  # two in front, one behind every third row
    for i in range(used):
        spread += [fa[i:i + 1]] + [off] * (i % 3 == 2)
    for what, new in (("behind", [fa] + [off] * 9), ("between", spread), ("both", spread + [off] * 3)):
        new = torch.cat(new).reshape(-1)
        other = md.clone()
        other[:new.numel()] = new
        got = _launch(prep, cu, other, new.numel() // _lib.FA_METADATA_SIZE)
        for a, b in zip(got, ref):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), what


@requires_gpu
@pytest.mark.parametrize("schedule", ["host", "device"])
@pytest.mark.parametrize("name,batch", [
    ("swa_decode_b32_h64", 3), ("mla_decode_b64_h128_k2048", 66),
    ("mla_fp8_decode_t128_h128_k2048", 3), ("swa_topk_decode_b32_h64_k512", 70)])
def test_no_sequence_has_a_row(name, batch, schedule):
    print(f"[gpu-rows-out-of-use] no rows: {name} batch={batch} {schedule}", flush=True)
    for lead, tail in ((0, 5), (4, 0), (2, 3)):
        t = _tnd(name, batch, [0] * batch, lead, tail)
        for _ in range(2):  # (the second call's output memory has been used)
            out, lse = sparse_attn_sharedkv(**t, schedule=schedule, return_softmax_lse=True)
            assert not out.any() and not lse.any()
            out.fill_(7.0)
            lse.fill_(7.0)
            del out, lse
