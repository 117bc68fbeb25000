"""Index arithmetic at odd geometries: block sizes and compression ratios that are not
powers of two (the kernels divide by multiplication), one-row blocks, ratios past the
context, lists that end at or just past a resolution's per-thread strides, on every
kernel, against the oracle (a wrongly gathered row moves an output by far more than the
tolerance: values are N(0, 1) * 0.5 over at most a few hundred rows)."""

import math

import pytest
import torch

from oracle.checks import check_strict
from oracle.golden_ref import sparse_attn_oracle

pytestmark = pytest.mark.gpu

HAS_GPU = torch.cuda.is_available()
requires_gpu = pytest.mark.skipif(not HAS_GPU, reason="needs a ROCm GPU")

if HAS_GPU:
    from sparse_attn_sharedkv_amd import quantize_kv_fp8, sparse_attn_sharedkv


def _pool(lens, bs, d, g):
    per = [max(-(-n // bs), 1) for n in lens]
    perm = torch.randperm(sum(per), generator=g).to(torch.int32)
    table = torch.full((len(lens), max(per)), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(per):
        table[b, :n] = perm[at:at + n]
        at += n
    return (torch.randn(sum(per), bs, 1, d, generator=g) * 0.5).to(torch.bfloat16), table


@requires_gpu
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("scenario,win,ratio,k,qlens,kvlens,heads,d,bs1,bs2", [
    (1, 127, 1, 0, [1, 1, 1], [129, 31, 500], 64, 576, 1, 1),
    (1, 255, 1, 0, [1, 1], [257, 256], 64, 512, 7, 1),       # 256 positions: one per thread
    (1, 319, 1, 0, [1, 1], [321, 319], 32, 576, 48, 1),      # 320: just past a stride
    (1, 5, 1, 0, [9, 3], [40, 3], 64, 512, 3, 1),            # row pairs
    (2, 63, 7, 0, [1, 1], [700, 64], 128, 512, 100, 13),
    (2, -1, 3, 0, [5, 4], [333, 200], 64, 576, 5, 11),
    (2, 31, 1000, 0, [2, 1], [300, 500], 16, 576, 33, 1),    # ratio past the context
    (3, 31, 5, 40, [1, 2], [400, 77], 64, 576, 9, 10),
    (3, -1, 1, 449, [1, 1], [450, 12], 128, 576, 17, 17),
    (3, 64, 3, 100, [30, 40], [500, 300], 128, 512, 31, 6),  # 128-head items (70 rows)
    (3, 64, 3, 100, [30, 40], [500, 300], 128, 576, 31, 6),
])
def test_odd_geometry(scenario, win, ratio, k, qlens, kvlens, heads, d, bs1, bs2, fp8):
    if fp8 and d != 576:
        pytest.skip("fp8 rows have 576 dims")
    print(f"[gpu-odd-geometry] scenario {scenario} win {win} ratio {ratio} blocks {bs1}/{bs2} "
          f"H={heads} d={d} fp8={fp8}", flush=True)
    g = torch.Generator().manual_seed(sum(kvlens) + bs1)
    n = sum(qlens)
    ori, t1 = _pool(kvlens, bs1, d, g)
    kw = dict(q=(torch.randn(n, heads, d, generator=g) * 0.5).to(torch.bfloat16), ori_kv=ori,
              ori_block_table=t1, seqused_kv=torch.tensor(kvlens, dtype=torch.int32),
              cu_seqlens_q=torch.tensor([0] + qlens).cumsum(0).to(torch.int32),
              sinks=torch.rand(heads, generator=g) * 2 - 1, softmax_scale=1 / math.sqrt(d),
              ori_win_left=win, layout_q="TND", head_dim_v=512)
    if scenario >= 2:
        cmp_, t2 = _pool([max(x // ratio, 1) for x in kvlens], bs2, d, g)
        kw.update(cmp_kv=cmp_, cmp_block_table=t2, cmp_ratio=ratio)
    if scenario == 3:
        idx = torch.full((n, 1, k), -1, dtype=torch.int32)
        t = 0
        for ql, kl in zip(qlens, kvlens):
            for s in range(ql):
                thr = max((kl - ql + s + 1) // ratio, 0)
                sel = torch.randperm(thr, generator=g)[:k]
                idx[t, 0, :sel.numel()] = sel.to(torch.int32)
                t += 1
        kw.update(cmp_sparse_indices=idx)
    dev = {a: (v.cuda() if isinstance(v, torch.Tensor) else v) for a, v in kw.items()}
    ref_kw = dict(kw)
    if fp8:
        from oracle.fp8_rows import dequantize_rows
        for name in ("ori_kv", "cmp_kv"):
            if name in kw:
                rows = quantize_kv_fp8(dev[name].reshape(-1, d))
                dev[name] = rows.view(*kw[name].shape[:-1], 656)
                deq = dequantize_rows(rows.cpu().numpy())
                ref_kw[name] = torch.as_tensor(deq).to(torch.bfloat16).view(kw[name].shape)
        dev["kv_cache_dtype"] = "fp8_ds_mla"
    ref, ref_lse = sparse_attn_oracle(**ref_kw)
    got = {}
    for how in ("host", "device"):
        out, lse = sparse_attn_sharedkv(**dev, schedule=how, return_softmax_lse=True)
        torch.cuda.synchronize()
        check_strict(out.cpu(), ref, lse.cpu(), ref_lse)
        got[how] = (out, lse)
    assert torch.equal(got["host"][0], got["device"][0])
    assert torch.equal(got["host"][1], got["device"][1])
