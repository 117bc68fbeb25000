"""Where captured calls get their arrival counters (``sas_merge_sync_take``): streams of one
capture never share an array, nor do captures; a process may make its first library call
inside a capture; and when every array is taken, captured calls zero one of their own.
Replays, with eager calls between them, are bitwise the eager call."""

import ctypes
import os
import subprocess
import sys

import pytest
import torch

from oracle import gen

pytestmark = pytest.mark.gpu

HAS_GPU = torch.cuda.is_available()
requires_gpu = pytest.mark.skipif(not HAS_GPU, reason="needs a ROCm GPU")

if HAS_GPU:
    from sparse_attn_sharedkv_amd import _lib, api


def _take(stream):
    return _lib.load().sas_merge_sync_take(ctypes.c_void_p(stream.cuda_stream))


@requires_gpu
def test_streams_of_one_capture_have_their_own():
    kws = [gen.build_workload("mla_decode_b64_h128_k2048", device="cuda", seed=s, batch=8)
           for s in (1, 2)]
    preps = [api.prepare(**kw, core_num=100, _m_base=128, _separate_merge=False) for kw in kws]
    refs = []
    for p in preps:
        api.launch(p)
        refs.append([p.out.clone(), p.lse.clone()])
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    graph, taken = torch.cuda.CUDAGraph(), {0: set(), 1: set()}
    with torch.cuda.graph(graph):
        main = torch.cuda.current_stream()
        side.wait_stream(main)
        for _ in range(3):  # calls of the two branches in turn
            api.launch(preps[0])
            taken[0].add(preps[0].args.merge_sync)
            with torch.cuda.stream(side):
                api.launch(preps[1])
            taken[1].add(preps[1].args.merge_sync)
        same = [_take(main), _take(main)]
        main.wait_stream(side)
    assert not taken[0] & taken[1], "two streams share an array"
    assert same[0] == same[1], "calls in a row on one stream share one"
    other = torch.cuda.CUDAGraph()
    with torch.cuda.graph(other):
        assert _take(torch.cuda.current_stream()) not in taken[0] | taken[1] | set(same)
        preps[0].out.zero_()
    assert not _take(torch.cuda.current_stream()), "not capturing: refused"
    for r in range(4):
        for p in preps:
            p.out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for p, ref in zip(preps, refs):
            assert torch.equal(p.out, ref[0]) and torch.equal(p.lse, ref[1]), r


# the captured call is the process's first; then one captured after every array is taken
CHILD = r"""
import ctypes, torch
from oracle import gen
from sparse_attn_sharedkv_amd import _lib, api, sparse_attn_sharedkv
kw = gen.build_workload("mla_decode_b64_h128_k2048", device="cuda", seed=3, batch=64)
call = lambda: sparse_attn_sharedkv(**kw, schedule="device", return_softmax_lse=True)
torch.cuda.synchronize()
assert _lib._lib is None, "the library is loaded already"

def capture():
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    return graph, out

def check(graph, out, what):
    for r in range(4):
        for t in out:
            t.fill_(float("nan"))
        graph.replay()
        eager = call()
        torch.cuda.synchronize()
        for a, b in zip(out, eager):
            assert torch.isfinite(b).all() and torch.equal(a, b), (what, r)
    print(what, "ok", flush=True)

first = capture()
assert not api._CAPTURED_MERGE_SYNC, "the first capture took no array of the library's"
check(*first, "first call in a capture")
lib, side, n = _lib.load(), torch.cuda.Stream(), 0
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    main = torch.cuda.current_stream()
    side.wait_stream(main)
    streams = [ctypes.c_void_p(s.cuda_stream) for s in (main, side)]
    seen = set()
    while n < 3000:
        at = lib.sas_merge_sync_take(streams[n % 2])
        if not at:
            break
        assert at not in seen, "an array given twice"
        seen.add(at)
        n += 1
    with torch.cuda.stream(side):
        torch.zeros(1, device="cuda")
    main.wait_stream(side)
    kw["sinks"].add_(0)
assert 500 < n < 1024, n
assert "every array is taken" in _lib.last_error()
last = capture()
assert len(api._CAPTURED_MERGE_SYNC) == 1
check(*last, "captured after every array was taken")
check(*first, "first capture again")
"""


@requires_gpu
def test_first_call_in_a_capture_and_every_array_taken():
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run([sys.executable, "-c", CHILD], cwd=root, capture_output=True, text=True,
                         timeout=110)
    print(res.stdout[-2000:], res.stderr[-2000:], flush=True)
    assert res.returncode == 0
    assert res.stdout.count("ok") == 3
