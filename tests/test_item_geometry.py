"""An item's geometry as the kernels form it (32 bits, division by multiplication)
against ``item_geom``, which both schedulers use: the same over lengths, rows, windows,
ratios and top-k widths from the smallest to the largest the entry points take, negative
windows among them. On the CPU: ``sas_items.h`` compiled for the host. And on the GPU,
windows below -1 through the C entry point: an empty window, as -1."""

import os
import shutil
import subprocess

import pytest
import torch

from oracle import gen
from sparse_attn_sharedkv_amd import _lib

CSRC = os.path.join(os.path.dirname(_lib.__file__), "csrc")
GXX = shutil.which("g++")
HIP_INCLUDE = "/opt/rocm/include"

PROGRAM = r"""
#include "sas_items.h"
#include <cstdio>
#include <cstdlib>
#include <climits>
#include <random>
static long n_bad = 0, n_all = 0;
static void check(int aq, int akv, int s, int wl, int scen, int ratio, int topk) {
  const sas::ItemGeom r = sas::item_geom(aq, akv, s, wl, scen, ratio, topk);
  const sas::ItemGeom g = sas::item_geom_div(aq, akv, s, wl, scen, sas::FastDiv::of(ratio), topk);
  ++n_all;
  if (r.n_win != g.n_win || r.thr != g.thr || r.n_cmp != g.n_cmp ||
      (r.n_win > 0 && r.win_lo != g.win_lo)) {
    if (n_bad++ < 5)
      printf("act_q %d act_kv %d s %d win %d scenario %d ratio %d topk %d: %d %d %d %d, not %d %d %d %d\n",
             aq, akv, s, wl, scen, ratio, topk, g.win_lo, g.n_win, g.thr, g.n_cmp, r.win_lo, r.n_win,
             r.thr, r.n_cmp);
  }
}
int main() {
  const int wins[] = {INT_MIN, INT_MIN + 1, -1000, -2, -1, 0, 1, 5, 127, 128, 1 << 20, INT_MAX};
  const int ratios[] = {1, 2, 3, 4, 5, 7, 16, 100, 127, 128, 1000, 65535, 1 << 30, INT_MAX};
  const int topks[] = {0, 1, 7, 512, 2048, INT_MAX};
  const int rows[] = {1, 2, 9, 640, 1 << 20};
  const int lens[] = {-3, 0, 1, 2, 8, 127, 128, 129, 640, 8192, 131072, (1 << 24) + 1, INT_MAX - 1, INT_MAX};
  for (int aq : rows)
    for (int akv : lens)
      for (int s : {0, 1, aq / 2, aq - 2, aq - 1})
        if (s >= 0 && s < aq)
          for (int wl : wins)
            for (int ratio : ratios)
              for (int topk : topks)
                for (int scen = 1; scen <= 3; ++scen) check(aq, akv, s, wl, scen, ratio, topk);
  std::mt19937 rng(1);
  auto any = [&](int lo, int hi) { return std::uniform_int_distribution<int>(lo, hi)(rng); };
  for (int i = 0; i < 2000000; ++i) {
    const int aq = any(1, 1 << any(0, 20));
    check(aq, any(-1, INT_MAX >> any(0, 30)), any(0, aq - 1), any(-2, INT_MAX >> any(0, 30)), any(1, 3),
          any(1, INT_MAX >> any(0, 30)), any(0, 4096));
  }
  printf("%ld of %ld\n", n_bad, n_all);
  return n_bad != 0;
}
"""


@pytest.mark.skipif(GXX is None or not os.path.isdir(HIP_INCLUDE), reason="needs g++ and HIP's headers")
def test_kernel_geometry_is_the_schedulers(tmp_path):
    (tmp_path / "geom.cpp").write_text(PROGRAM)
    subprocess.run([GXX, "-O1", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I", CSRC,
                    "-I", HIP_INCLUDE, "geom.cpp", "-o", "geom"], cwd=tmp_path, check=True)
    res = subprocess.run([str(tmp_path / "geom")], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout + res.stderr


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a ROCm GPU")
@pytest.mark.parametrize("name,batch,cores", [
    ("topk_decode_b2_h16_k256", 2, 3), ("mla_decode_b64_h128_k2048", 3, 64),
    ("mla_mtp_decode_b64_h128_k2048", 40, 256), ("mla_fp8_decode_t128_h128_k2048", 3, 64),
    ("cfa_prefill_t8192_h64", 1, 256),
])
def test_windows_below_minus_one_are_empty(name, batch, cores):
    from sparse_attn_sharedkv_amd import api
    print(f"[gpu-item-geometry] {name}", flush=True)
    kw = gen.build_workload(name, device="cuda", seed=2, batch=batch, ctx_override=[900] * batch)
    kw["ori_win_left"] = -1
    if kw["layout_q"] == "TND" and kw["q"].shape[0] > 900:  # (prefill: 900 rows)
        kw["q"] = kw["q"][:900].contiguous()
        kw["cu_seqlens_q"] = torch.tensor([0, 900], dtype=torch.int32, device="cuda")
    prep = api.prepare(**kw, core_num=cores)
    api.launch(prep)
    ref = [prep.out.clone(), prep.lse.clone()]
    for win in (-2, -70, -2**31):
        prep.args.ori_win_left = win
        prep.out.fill_(7.0)
        api.launch(prep)
        torch.cuda.synchronize()
        for a, b in zip((prep.out, prep.lse), ref):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), win
