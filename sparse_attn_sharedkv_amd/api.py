"""Host entry point ``sparse_attn_sharedkv`` (signature and behaviour of api.py:129-397).

Scenario detection (api.py:196-202):

* ``cmp_kv=None, cmp_sparse_indices=None`` -> SWA (scenario 1)
* ``cmp_kv=<tensor>, cmp_sparse_indices=None`` -> CFA (scenario 2)
* ``cmp_kv=<tensor>, cmp_sparse_indices=<tensor>`` -> SCFA (scenario 3)

Q / indices are flattened to ``[total_tokens, ...]`` with a per-batch
``q_prefix`` exactly as api.py:208-240 does (TND passes through, BSND is a
free reshape). The paged caches go to the GPU untouched; the HIP kernels
resolve block tables on the device. Additions over the reference, all
optional and defaulting to its behaviour: ``head_dim_v`` (output width; the
first ``head_dim_v`` columns of each shared row are V, as in MLA where
d_qk = 576 and d_v = 512), head counts other than 64 (multiples of 16 up
to 128), and ``kv_cache_dtype`` (``"fp8_ds_mla"``: 656-byte fp8 rows, see
``kv_fp8``; by default inferred from the cache tensor's dtype).

Errors follow the reference: AssertionError for unsupported masks / layouts,
missing ``cu_seqlens_q`` in TND, top-k length mismatch and metadata size;
ValueError for dtypes and shapes; RuntimeError (with the library's message)
for launch failures. Everything is checked on the host before any launch.
"""

from __future__ import annotations

import collections
import ctypes
import functools
import threading
from dataclasses import dataclass, field
from typing import Optional, Tuple, Union

import torch

from . import _lib
from .metadata import (AIC_CORE_NUM, CFG_OFFSET, DEFAULT_CORE_NUM,  # noqa: F401
                       DEFAULT_MIN_SPLIT_BLOCKS, DEFAULT_S2_BASE, FD_METADATA_SIZE, FD_OFFSET, SAS_META_SIZE,
                       build_metadata, build_metadata_device, config_row, m_base_for,
                       m_base_valid)

DEFAULT_BLOCK_I = 128  # kernel.py:65, kept for callers that import it
SUPPORTED_HEAD_DIMS = (512, 576)
SUPPORTED_HEAD_DIM_V = (512,)
FP8_CACHE_DTYPES = (torch.uint8, torch.float8_e4m3fn)


def _kv_format(kv_cache_dtype: Optional[str], ori_kv: torch.Tensor) -> int:
    """Row format of the caches: native (q's dtype) or the 656-byte fp8 rows."""
    if kv_cache_dtype in (None, "auto"):
        return _lib.KV_FP8_DS_MLA if ori_kv.dtype in FP8_CACHE_DTYPES else _lib.KV_NATIVE
    if kv_cache_dtype == "fp8_ds_mla":
        return _lib.KV_FP8_DS_MLA
    raise ValueError(f"unsupported kv_cache_dtype {kv_cache_dtype!r} "
                     "(None, 'auto' or 'fp8_ds_mla')")


def _dtype_code(t: torch.dtype) -> int:
    if t == torch.bfloat16:
        return _lib.DTYPE_BF16
    if t == torch.float16:
        return _lib.DTYPE_FP16
    raise ValueError(f"unsupported torch dtype {t}")


@dataclass
class Prepared:
    """A fully validated call: device tensors, launch arguments, output views."""

    args: _lib.SasAttnArgs
    keep: list = field(default_factory=list)   # tensors that must outlive the launch
    out: Optional[torch.Tensor] = None
    lse: Optional[torch.Tensor] = None
    layout_q: str = "TND"
    bsnd_shape: Optional[tuple] = None
    device: Optional[torch.device] = None
    q_lens: int = _lib.QLENS_ARRAYS  # form of the query row counts (sas_attention_launch_lens)
    phase_bits: int = 0    # kernel-form bits every launch of this call carries (SAS_PHASE_FP8_QK)
    merge_in_kernel: bool = True  # split items merged by their last piece (SasAttnArgs.merge_sync)


# Split items are merged inside the attention kernel (by the piece that finishes
# last) when no item has more than this many pieces; with more, the merge kernel
# spreads the merging over all compute units and is faster, although it is a second
# launch, or a second node of a graph. Measured on MI355X, us, merge kernel / inside,
# replays of a graph of one call (calls in a row): MLA decode 64 x 128 heads, 2 pieces,
# 69.2 / 66.6 (63.7 / 62.0); in 128-head items, 4 pieces, 70.2 / 70.9 (65.6 / 65.1);
# window + top-k decode of 64 sequences, 3 pieces, 32.4 / 35.3 (28.0 / 30.5), of 32,
# 5 pieces, 24.9 / 29.7 (20.6 / 25.0); MLA decode 32 x 128 heads, 8 pieces,
# 50.8 / 55.5 (46.1 / 50.7).
MERGE_IN_KERNEL_MAX_PIECES = 2


def _max_pieces(md: torch.Tensor) -> int:
    """Largest piece count of a split item in a host schedule (0: nothing split)."""
    cfg = md[CFG_OFFSET:CFG_OFFSET + 8].tolist()
    nfd = int(cfg[3])
    if nfd <= 0:
        return 0
    fd = md[FD_OFFSET:FD_OFFSET + nfd * FD_METADATA_SIZE].view(nfd, FD_METADATA_SIZE)
    return int(fd[:, 4].max().item())


@functools.lru_cache(maxsize=64)
def _cached_schedule(act_q: tuple, act_kv: tuple, num_heads: int, ori_win_left: int,
                     scenario: int, cmp_ratio: int, topk: int, core_num: int,
                     item64: bool, m_base: Optional[int] = None) -> Tuple[torch.Tensor, int]:
    md = build_metadata(act_q=act_q, act_kv=act_kv, num_heads=num_heads,
                        ori_win_left=ori_win_left, scenario=scenario, cmp_ratio=cmp_ratio,
                        cmp_topk=topk, core_num=core_num, item64=item64, m_base=m_base)
    return md, _max_pieces(md)


# Between a host-scheduled call's lengths arriving and its launch the GPU waits, so
# prepare() reads the lengths back behind the rest of its work, and the cached host
# schedules are kept on the GPU they were used on, by their inputs: a call whose
# lengths give a known one does not copy its 64 KB again. Calls of 8192 query rows in
# a row, 64 heads, on one MI355X: window-only 449 -> 409 us, dense pool 482 -> 426,
# top-k 1143 -> 1078, with the kernels' own 384, 402 and 1069. (Lengths new on every
# call, two sequences cut elsewhere each time, against one cut repeated: 521 against
# 413 us window-only, 550 against 427, 1172 against 1032. The on-device
# scheduler instead was slower: such schedules, of more than ~4000 items, are rebuilt
# on each call, 120 us.) An entry is complete before it is handed out, so any stream
# may read it; a use on another stream than its own is recorded, so that an evicted
# one is not given out again under a kernel that still reads it.
_GPU_SCHEDULES: "collections.OrderedDict" = collections.OrderedDict()
_GPU_SCHEDULES_MAX = 64
_GPU_SCHEDULES_LOCK = threading.Lock()


def _schedule_on(dev: torch.device, key: tuple, md: torch.Tensor) -> torch.Tensor:
    st = torch.cuda.current_stream(dev)
    with _GPU_SCHEDULES_LOCK:
        hit = _GPU_SCHEDULES.get((dev, key))
        if hit is not None:
            _GPU_SCHEDULES.move_to_end((dev, key))
    if hit is None:
        hit = (md.to(dev), st.cuda_stream)
        st.synchronize()
        with _GPU_SCHEDULES_LOCK:
            _GPU_SCHEDULES[(dev, key)] = hit
            while len(_GPU_SCHEDULES) > _GPU_SCHEDULES_MAX:
                _GPU_SCHEDULES.popitem(last=False)
    if hit[1] != st.cuda_stream:
        hit[0].record_stream(st)
    return hit[0]


# Schedules built by the on-device scheduler for calls without ``metadata``: one
# library-owned buffer per (device, stream), written only by that scheduler on
# that stream, so an unchanged schedule is kept instead of rebuilt. Calls on one
# stream run in order; different streams get different buffers.
# A call captured into a HIP graph gets a buffer of its own instead (graphs
# captured on one stream may be replayed on different streams, or beside eager
# calls on the capture stream, so a shared buffer would race); it is allocated
# from the capture's pool and kept for the life of the process, because every
# replay of the graph reads and writes it. Its first replay builds the schedule,
# later replays keep it while the lengths give the same schedule.
_DEVICE_SCHEDULES: dict = {}
_CAPTURED_SCHEDULES: list = []
_DEVICE_SCHEDULES_LOCK = threading.Lock()


def _schedule_buffer(dev: torch.device) -> torch.Tensor:
    if torch.cuda.is_current_stream_capturing():
        buf = torch.empty(SAS_META_SIZE, dtype=torch.int32, device=dev)
        with _DEVICE_SCHEDULES_LOCK:
            _CAPTURED_SCHEDULES.append(buf)
        return buf
    st = torch.cuda.current_stream(dev)
    key = (dev.index, st.cuda_stream)
    with _DEVICE_SCHEDULES_LOCK:
        buf = _DEVICE_SCHEDULES.get(key)
        if buf is None:
            buf = torch.zeros(SAS_META_SIZE, dtype=torch.int32, device=dev)
            _DEVICE_SCHEDULES[key] = buf
    return buf


# Arrival counters of the split-KV merge done inside the attention kernel
# (SasAttnArgs.merge_sync): zero at rest, one buffer per (device, stream) so that
# calls on different streams never share one. Calls captured into a HIP graph take
# one of the library's own zeroed arrays (sas_merge_sync_take: calls that follow one
# another on one stream of a capture share one, taken for the life of the process);
# when those are all taken, a buffer zeroed by a fill kernel recorded in the graph.
_MERGE_SYNC: dict = {}
_CAPTURED_MERGE_SYNC: list = []


def _captured_merge_sync(dev: torch.device, st: torch.cuda.Stream) -> int:
    """Address of the counters for a call being captured on ``st``."""
    with torch.cuda.device(dev):
        at = _lib.load().sas_merge_sync_take(ctypes.c_void_p(st.cuda_stream))
    if at:
        return at
    buf = torch.zeros(_lib.MERGE_SYNC_WORDS, dtype=torch.int64, device=dev)
    with _DEVICE_SCHEDULES_LOCK:
        _CAPTURED_MERGE_SYNC.append(buf)
    return buf.data_ptr()


def _merge_sync_buffer(dev: torch.device, st: torch.cuda.Stream) -> torch.Tensor:
    key = (dev.index, st.cuda_stream)
    with _DEVICE_SCHEDULES_LOCK:
        buf = _MERGE_SYNC.get(key)
        if buf is None:
            buf = torch.zeros(_lib.MERGE_SYNC_WORDS, dtype=torch.int64, device=dev)
            _MERGE_SYNC[key] = buf
    return buf


def _ptr(t: Optional[torch.Tensor]):
    return t.data_ptr() if t is not None else None


def _read_back(ts):
    """int32 tensors on one GPU on their way to the host: ``(pinned words, event)``."""
    host = torch.empty(sum(t.numel() for t in ts), dtype=torch.int32, pin_memory=True)
    at = 0
    for t in ts:
        host[at:at + t.numel()].copy_(t, non_blocking=True)
        at += t.numel()
    done = torch.cuda.Event()
    done.record(torch.cuda.current_stream(ts[0].device))
    return host, done


def prepare(q: torch.Tensor, *, ori_kv: torch.Tensor, cmp_kv: Optional[torch.Tensor] = None,
            cmp_sparse_indices: Optional[torch.Tensor] = None, ori_block_table: torch.Tensor,
            cmp_block_table: Optional[torch.Tensor] = None,
            cu_seqlens_q: Optional[torch.Tensor] = None,
            seqused_q: Optional[torch.Tensor] = None, seqused_kv: torch.Tensor,
            sinks: torch.Tensor, metadata: Optional[torch.Tensor] = None,
            softmax_scale: float, cmp_ratio: Optional[int] = None, ori_mask_mode: int = 4,
            cmp_mask_mode: int = 3, ori_win_left: int = 127, ori_win_right: int = 0,
            layout_q: str = "TND", layout_kv: str = "PA_ND",
            core_num: int = DEFAULT_CORE_NUM, topk_cmp: Optional[int] = None,
            head_dim_v: Optional[int] = None,
            kv_cache_dtype: Optional[str] = None,
            schedule: Optional[str] = None,
            fp8_qk: bool = False,
            _stream_schedule: bool = False,
            _pipelined: bool = False, _separate_merge: Optional[bool] = None,
            _m_base: Optional[int] = None, _row_items: bool = False) -> Prepared:
    """Validate and stage one call (host work of api.py:186-384) without launching.

    ``schedule``: ``"host"`` reads the lengths back and schedules on the CPU (the
    reference's behaviour, api.py:335-360); ``"device"`` keeps them on the GPU and
    runs the on-device scheduler (no host synchronisation); ``None`` means
    ``"device"`` when ``metadata`` is a GPU tensor (it is then not read back) and
    ``"host"`` otherwise. ``_stream_schedule`` (for callers that launch right after
    preparing, on the same stream): a device-built schedule goes to the library's
    buffer for the current stream and is kept when unchanged; otherwise every
    prepared call schedules into a buffer of its own. ``_pipelined`` (tests): native
    rows run through the kernel fp8 rows use (``SAS_PHASE_PIPELINED``, items of at
    most 64 heads), for bitwise comparisons with the fp8 path. ``_separate_merge``
    (tests, timing): True merges split items by the merge kernel after the attention
    kernel, False inside it; None (default) inside it when no item has more than
    ``MERGE_IN_KERNEL_MAX_PIECES`` pieces. ``_m_base`` (tests, timing): heads per item instead
    of ``m_base_for``'s choice (a call with its own ``metadata`` uses the metadata's).
    ``_row_items`` (tests, timing): one query row per workgroup item even where the
    library would pair consecutive rows (``SAS_PHASE_ROW_ITEMS``).
    """
    del seqused_q  # API-parity placeholder (api.py:186)
    assert ori_mask_mode == 4, "only ori_mask_mode=4 supported"
    assert cmp_mask_mode == 3 or cmp_kv is None, "only cmp_mask_mode=3 supported"
    assert ori_win_right == 0, "only ori_win_right=0 supported"
    assert layout_kv == "PA_ND", "only layout_kv=PA_ND supported"
    assert layout_q in ("TND", "BSND"), f"unsupported layout_q={layout_q!r}"

    if schedule not in (None, "host", "device"):
        raise ValueError(f"schedule must be 'host' or 'device', got {schedule!r}")
    use_dev = schedule == "device" or (
        schedule is None and metadata is not None and metadata.device.type == "cuda")
    dtype = q.dtype
    dcode = _dtype_code(dtype)
    if cmp_kv is None:
        scenario = 1
    elif cmp_sparse_indices is None:
        scenario = 2
    else:
        scenario = 3

    # ---- flatten Q / indices to [total_tokens, ...] (api.py:208-240) ----
    cu_host = None
    # lengths read back for a host schedule: late, behind the rest of the preparation
    late = (_stream_schedule and metadata is None and not use_dev and q.is_cuda
            and seqused_kv.is_cuda and seqused_kv.dim() == 1 and seqused_kv.numel() > 0
            and not torch.cuda.is_current_stream_capturing())
    if layout_q == "TND":
        assert cu_seqlens_q is not None, "cu_seqlens_q is required for TND"
        if q.dim() != 3:
            raise ValueError(f"TND q must be [T, N1, D], got {tuple(q.shape)}")
        t1, n1, d = q.shape
        total = t1
        # the launch takes cu_seqlens_q itself (QLENS_CUMULATIVE below): the host needs
        # it for the schedule only
        late = late and t1 > 0 and cu_seqlens_q.dim() == 1 and cu_seqlens_q.numel() > 1 \
            and cu_seqlens_q.is_cuda
        if use_dev or late:
            # lengths stay on the GPU; rows past cu_seqlens_q[-1] are zero-filled
            nb = cu_seqlens_q.numel() - 1
            act_q = prefix = None
            padded = True
        else:
            cu_host = [int(x) for x in cu_seqlens_q.to(torch.int32).cpu().tolist()]
            nb = len(cu_host) - 1
            act_q = [cu_host[i + 1] - cu_host[i] for i in range(nb)]
            prefix = cu_host[:-1]
            padded = (cu_host[-1] != t1) if cu_host else t1 > 0
    else:
        if q.dim() != 4:
            raise ValueError(f"BSND q must be [B, S, N1, D], got {tuple(q.shape)}")
        nb, s_max, n1, d = q.shape
        total = nb * s_max
        prefix = [i * s_max for i in range(nb)]
        act_q = [s_max] * nb
        padded = False
        late = late and cu_seqlens_q is None and total > 0
        if cu_seqlens_q is not None and use_dev:
            act_q = None
            padded = True
        elif cu_seqlens_q is not None:
            cu_host = [int(x) for x in cu_seqlens_q.to(torch.int32).cpu().tolist()]
            act_q = [cu_host[i + 1] - cu_host[i] for i in range(nb)]
            padded = any(a != s_max for a in act_q)

    idx_flat = None
    k = 0
    if scenario == 3:
        ci = cmp_sparse_indices
        if ci.dim() != (3 if layout_q == "TND" else 4):
            raise ValueError(f"cmp_sparse_indices has rank {ci.dim()} for layout {layout_q}")
        idx_flat = ci.reshape(total, ci.shape[-2], ci.shape[-1])
        n2 = idx_flat.shape[1]
        k = topk_cmp if topk_cmp is not None else idx_flat.shape[2]
        assert k == idx_flat.shape[2], "topk_cmp does not match cmp_sparse_indices last dim"
    elif scenario == 2:
        n2 = cmp_kv.shape[2]
    else:
        n2 = ori_kv.shape[2]

    kv_fmt = _kv_format(kv_cache_dtype, ori_kv)
    fp8_rows = kv_fmt == _lib.KV_FP8_DS_MLA
    # items of at most 64 heads: the fp8 Q·Kᵀ form and the pipelined kernel (m_base_for)
    item64 = _pipelined
    # the item size: by query rows for a schedule this call builds, by sequences
    # for one it is handed (the count its builder used, m_base_for)
    m_base = (m_base_for(int(n1), item64, nb, fp8_rows,
                         rows=int(total) if metadata is None else None)
              if _m_base is None else int(_m_base))
    if not m_base_valid(int(n1), item64, m_base):
        raise ValueError(f"no kernel for items of {m_base} heads at {n1} heads")
    row_width = _lib.FP8_ROW_BYTES if fp8_rows else d
    dv = (512 if fp8_rows else d) if head_dim_v is None else int(head_dim_v)
    if n2 != 1 or ori_kv.shape[2] != 1 or ori_kv.shape[-1] != row_width:
        raise ValueError(f"only N2=1 shared KV with KV width == q width supported "
                         f"(got N2={n2}, q D={d}, kv {tuple(ori_kv.shape)})")
    if d not in SUPPORTED_HEAD_DIMS or dv not in SUPPORTED_HEAD_DIM_V or dv > d:
        raise ValueError(f"supported head dims: D in {SUPPORTED_HEAD_DIMS} with head_dim_v in "
                         f"{SUPPORTED_HEAD_DIM_V} (got D={d}, head_dim_v={dv})")
    if n1 < 16 or n1 > 128 or n1 % 16 != 0:
        raise ValueError(f"N1 must be a multiple of 16 in [16, 128] (got N1={n1})")
    if fp8_rows:
        if d != 576 or dtype != torch.bfloat16:
            raise ValueError("fp8_ds_mla caches need bf16 queries with D=576")
        for t in (ori_kv, cmp_kv):
            if t is not None and t.dtype not in FP8_CACHE_DTYPES:
                raise ValueError("fp8_ds_mla caches are uint8 or float8_e4m3fn tensors "
                                 f"[blocks, block_size, 1, {_lib.FP8_ROW_BYTES}]")
    elif ori_kv.dtype != dtype or (cmp_kv is not None and cmp_kv.dtype != dtype):
        raise ValueError("KV caches must have q's dtype")
    if fp8_qk and not fp8_rows:
        raise ValueError("fp8_qk needs fp8_ds_mla cache rows")
    if ori_win_left < -1:
        raise ValueError("ori_win_left must be >= -1")
    if scenario >= 2:
        if cmp_block_table is None:
            raise ValueError("cmp_block_table is required with cmp_kv")
        if cmp_ratio is not None and cmp_ratio < 1:
            raise ValueError("cmp_ratio must be >= 1")
        if cmp_kv.shape[-1] != row_width or cmp_kv.shape[2] != 1:
            raise ValueError("cmp_kv must be [blocks, block_size, 1, D]")
    cmp_ratio_eff = int(cmp_ratio) if cmp_ratio is not None else 4  # api.py:287
    if metadata is not None:
        assert metadata.numel() == SAS_META_SIZE, (
            f"metadata must have {SAS_META_SIZE} int32 entries (got {metadata.numel()})")
    # the kernels read seqused_kv[b] and block-table row b for every batch b
    if seqused_kv.numel() < nb:
        raise ValueError(f"seqused_kv has {seqused_kv.numel()} entries for {nb} sequences")
    if ori_block_table.dim() != 2 or ori_block_table.shape[0] < nb:
        raise ValueError(f"ori_block_table must be [>= {nb}, table_len] "
                         f"(got {tuple(ori_block_table.shape)})")
    if scenario >= 2 and (cmp_block_table.dim() != 2 or cmp_block_table.shape[0] < nb):
        raise ValueError(f"cmp_block_table must be [>= {nb}, table_len] "
                         f"(got {tuple(cmp_block_table.shape)})")

    dev = q.device
    if dev.type != "cuda":
        raise RuntimeError("sparse_attn_sharedkv runs on a ROCm GPU; q is on " + str(dev))

    # ---- query rows and lengths ----
    i32 = torch.int32
    seqused = seqused_kv.to(device=dev, dtype=i32).contiguous()
    # Callers that launch right after preparing hand the kernels cu_seqlens_q itself,
    # or nothing when every batch has as many rows, instead of arrays made from them
    q_lens = _lib.QLENS_ARRAYS
    act_q_d = cu_d = None
    if _stream_schedule and nb > 0 and total > 0:
        if layout_q == "TND":
            q_lens = _lib.QLENS_CUMULATIVE
            q_prefix = cu_d = cu_seqlens_q.to(device=dev, dtype=i32).reshape(-1).contiguous()
            padded = False  # (the kernels zero the rows of no batch)
        elif cu_seqlens_q is None:
            q_lens = _lib.QLENS_UNIFORM
            q_prefix = None
    # ---- device tensors ----
    q_flat = q.reshape(total, n1, d).contiguous()
    ori_kv_d = ori_kv.contiguous()
    ori_bt = ori_block_table.to(device=dev, dtype=i32).contiguous()
    cmp_kv_d = cmp_kv.contiguous() if cmp_kv is not None else None
    cmp_bt = cmp_block_table.to(device=dev, dtype=i32).contiguous() if cmp_kv is not None else None
    idx_d = idx_flat.to(device=dev, dtype=i32).contiguous() if idx_flat is not None else None
    if not use_dev and q_lens == _lib.QLENS_ARRAYS:
        q_prefix = torch.tensor(prefix, dtype=i32).to(dev, non_blocking=True)
        act_q_d = torch.tensor(act_q, dtype=i32).to(dev, non_blocking=True)
    sinks_d = sinks.to(device=dev, dtype=torch.float32).contiguous()
    if sinks_d.numel() != n1:
        raise ValueError(f"sinks must have N1={n1} entries")
    alloc = torch.zeros if padded else torch.empty
    out = alloc((total, n1, dv), dtype=dtype, device=dev)
    lse = alloc((total, n1), dtype=torch.float32, device=dev)
    for t in (q_flat, ori_kv_d, cmp_kv_d):
        if t is not None and t.device != dev:
            raise ValueError("all tensors must be on q's device")

    lens = None
    if late:
        lens = _read_back([cu_d, seqused] if layout_q == "TND" else [seqused])

    a = _lib.SasAttnArgs()
    a.q, a.ori_kv, a.ori_block_table = _ptr(q_flat), _ptr(ori_kv_d), _ptr(ori_bt)
    a.cmp_kv, a.cmp_block_table, a.cmp_indices = _ptr(cmp_kv_d), _ptr(cmp_bt), _ptr(idx_d)
    a.seqused_kv = _ptr(seqused)
    a.sinks, a.out, a.lse = _ptr(sinks_d), _ptr(out), _ptr(lse)
    a.batch, a.total_tokens, a.num_heads = nb, total, n1
    a.head_dim, a.head_dim_v = d, dv
    a.ori_block_num, a.ori_block_size, a.ori_table_len = (
        ori_kv_d.shape[0], ori_kv_d.shape[1], ori_bt.shape[1])
    if cmp_kv_d is not None:
        a.cmp_block_num, a.cmp_block_size, a.cmp_table_len = (
            cmp_kv_d.shape[0], cmp_kv_d.shape[1], cmp_bt.shape[1])
    a.topk = int(k)
    a.scenario, a.cmp_ratio, a.ori_win_left, a.dtype = scenario, cmp_ratio_eff, ori_win_left, dcode
    a.softmax_scale = float(softmax_scale)
    a.kv_format = kv_fmt

    # ---- schedule (api.py:335-366) ----
    if use_dev:
        # per-batch query rows and first flat token, computed on the GPU
        if q_lens != _lib.QLENS_ARRAYS:
            pass
        elif layout_q == "TND":
            cu_d = cu_seqlens_q.to(device=dev, dtype=i32).reshape(-1)
            act_q_d = (cu_d[1:] - cu_d[:-1]).contiguous()
            q_prefix = cu_d[:-1].contiguous()
        else:
            q_prefix = torch.arange(nb, dtype=i32, device=dev) * (total // max(nb, 1))
            if cu_seqlens_q is not None:
                cu_d = cu_seqlens_q.to(device=dev, dtype=i32).reshape(-1)
                act_q_d = (cu_d[1:] - cu_d[:-1]).contiguous()
            else:
                act_q_d = torch.full((nb,), total // max(nb, 1), dtype=i32, device=dev)
        if metadata is None:
            metadata_dev = build_metadata_device(
                batch=nb, act_q=act_q_d, cu_q=cu_d if act_q_d is None else None,
                uniform_q=total // max(nb, 1), act_kv=seqused, num_heads=int(n1),
                ori_win_left=int(ori_win_left), scenario=scenario, cmp_ratio=cmp_ratio_eff,
                cmp_topk=int(k), core_num=int(core_num),
                out=_schedule_buffer(dev) if _stream_schedule else None, item64=item64,
                m_base=m_base)
        else:
            metadata_dev = metadata.to(device=dev, dtype=i32).reshape(SAS_META_SIZE).contiguous()
        # capacities; the kernels read the schedule's own summary on the GPU. A
        # schedule supplied on the GPU may have been built for any core count up to
        # AIC_CORE_NUM, which this call cannot read without a host sync: launch for
        # that many workgroups (the unused ones exit at once) and size the workspace
        # for the most partial pieces such a schedule can have (two per core).
        cap = int(core_num) if metadata is None else AIC_CORE_NUM
        cfg = dict(num_fa=cap, num_fd=_lib.SCHED_DEVICE, num_partial_slots=2 * cap,
                   s2_base=DEFAULT_S2_BASE, m_base=m_base)
        # pieces per item are not known on the host: expect at most two when the
        # items are at least half as many as the workgroups, or when the longest
        # possible list has too few blocks for more
        items = total * ((n1 + cfg["m_base"] - 1) // cfg["m_base"])
        longest = int(ori_win_left) + 1
        if scenario == 3:
            longest += int(k)
        elif scenario == 2:
            longest += cmp_block_table.shape[1] * cmp_kv.shape[1]
        most = -(-longest // DEFAULT_S2_BASE) // DEFAULT_MIN_SPLIT_BLOCKS
        few_pieces = (int(core_num) <= MERGE_IN_KERNEL_MAX_PIECES * items
                      or most <= MERGE_IN_KERNEL_MAX_PIECES)
    elif metadata is None:
        if lens is not None:  # everything else is ready: from here to the launch the GPU waits
            lens[1].synchronize()
            words = lens[0].tolist()
            kv_host = tuple(words[-seqused.numel():])
            if layout_q == "TND":
                act_q = [b - a for a, b in zip(words[:nb], words[1:nb + 1])]
        else:
            kv_host = tuple(int(x) for x in seqused_kv.to(torch.int32).cpu().tolist())
        key = (tuple(act_q), kv_host, int(n1), int(ori_win_left), scenario, cmp_ratio_eff, int(k),
               int(core_num), item64, m_base)
        md, max_pieces = _cached_schedule(*key)
        cfg = config_row(md)
        metadata_dev = (_schedule_on(dev, key, md) if lens is not None
                        else md.to(dev, non_blocking=True))
        few_pieces = max_pieces <= MERGE_IN_KERNEL_MAX_PIECES
    else:
        metadata_dev = metadata.to(dev).to(torch.int32).reshape(SAS_META_SIZE).contiguous()
        cfg = config_row(metadata)  # host read of the schedule summary row
        few_pieces = _max_pieces(metadata.to("cpu", torch.int32).reshape(-1)) <= \
            MERGE_IN_KERNEL_MAX_PIECES
        assert cfg["num_heads"] == n1 and m_base_valid(n1, item64, cfg["m_base"]), (
            "metadata was built for a different head count or cache row format "
            "(fp8 cache rows: sparse_attn_sharedkv_metadata(..., kv_cache_dtype='fp8_ds_mla'))")
    ws = None
    if cfg["num_fd"] > 0 or use_dev:
        nbytes = _lib.load().sas_workspace_bytes(cfg["num_partial_slots"], cfg["m_base"], dv)
        ws = torch.empty(nbytes // 4, dtype=torch.float32, device=dev)

    a.q_prefix, a.act_q_lens = _ptr(q_prefix), _ptr(act_q_d)
    a.metadata, a.workspace = _ptr(metadata_dev), _ptr(ws)
    a.num_fa, a.num_fd = cfg["num_fa"], cfg["num_fd"]
    a.num_partial_slots, a.s2_base, a.m_base = (
        cfg["num_partial_slots"], cfg["s2_base"], cfg["m_base"])
    keep = [q_flat, ori_kv_d, ori_bt, cmp_kv_d, cmp_bt, idx_d, q_prefix, act_q_d, seqused,
            sinks_d, metadata_dev, out, lse, ws]
    return Prepared(args=a, keep=keep, out=out, lse=lse, layout_q=layout_q,
                    bsnd_shape=None if layout_q == "TND" else (nb, total // max(nb, 1), n1, dv),
                    device=dev, q_lens=q_lens, phase_bits=(_lib.SAS_PHASE_FP8_QK if fp8_qk else 0) |
                    (_lib.SAS_PHASE_PIPELINED if _pipelined else 0) |
                    (_lib.SAS_PHASE_ROW_ITEMS if _row_items else 0),
                    merge_in_kernel=few_pieces if _separate_merge is None
                    else not _separate_merge)


def uses_row_pairs(prep: Prepared) -> bool:
    """Whether the library runs this call as row pairs (two consecutive query rows
    of 64 heads per workgroup on the 128-head kernel; pieces of split items run
    alone): the rule of the library's launch (native rows, items of 64 heads with
    at most 64 heads, scenarios 1 and 2, several query rows in some sequence)."""
    a = prep.args
    return (a.kv_format == _lib.KV_NATIVE and a.m_base == 64 and a.num_heads <= 64
            and a.scenario <= 2 and a.total_tokens > a.batch
            and not (prep.phase_bits & (_lib.SAS_PHASE_ROW_ITEMS | _lib.SAS_PHASE_PIPELINED)))


def launch(prep: Prepared, stream: Optional[torch.cuda.Stream] = None, phases: int = 0) -> None:
    """Enqueue the attention (+ merge) kernels on ``stream`` (default: current stream).

    ``phases``: 0 both kernels, 1 the attention kernel only, 2 the merge only
    (a caller timing the two kernels separately enqueues 1 then 2).
    """
    lib = _lib.load()
    st = stream if stream is not None else torch.cuda.current_stream(prep.device)
    prep.args.phases = int(phases) | prep.phase_bits
    if not (prep.merge_in_kernel and prep.args.workspace):
        prep.args.merge_sync = None
    elif torch.cuda.is_current_stream_capturing():
        prep.args.merge_sync = _captured_merge_sync(prep.device, st)
    else:
        sync = _merge_sync_buffer(prep.device, st)
        prep.args.merge_sync = sync.data_ptr()
        if not any(t is sync for t in prep.keep):
            prep.keep.append(sync)
    rc = lib.sas_attention_launch_lens(ctypes.byref(prep.args), prep.q_lens,
                                       ctypes.c_void_p(st.cuda_stream))
    if rc != _lib.SAS_OK:
        raise RuntimeError(_lib.last_error())


def finalize(prep: Prepared, return_softmax_lse: bool):
    """Restore the caller's layout (api.py:386-397)."""
    out, lse = prep.out, prep.lse
    if prep.layout_q == "BSND":
        b, s, n1, dv = prep.bsnd_shape
        out = out.reshape(b, s, n1, dv)
        lse = lse.reshape(b, s, n1)
    if return_softmax_lse:
        return out, lse
    return out


def sparse_attn_sharedkv(
    q: torch.Tensor,
    *,
    ori_kv: torch.Tensor,
    cmp_kv: Optional[torch.Tensor] = None,
    cmp_sparse_indices: Optional[torch.Tensor] = None,
    ori_block_table: torch.Tensor,
    cmp_block_table: Optional[torch.Tensor] = None,
    cu_seqlens_q: Optional[torch.Tensor] = None,
    seqused_q: Optional[torch.Tensor] = None,
    seqused_kv: torch.Tensor,
    sinks: torch.Tensor,
    metadata: Optional[torch.Tensor] = None,
    softmax_scale: float,
    cmp_ratio: Optional[int] = None,
    ori_mask_mode: int = 4,
    cmp_mask_mode: int = 3,
    ori_win_left: int = 127,
    ori_win_right: int = 0,
    layout_q: str = "TND",
    layout_kv: str = "PA_ND",
    return_softmax_lse: bool = False,
    core_num: int = DEFAULT_CORE_NUM,
    topk_cmp: Optional[int] = None,
    head_dim_v: Optional[int] = None,
    kv_cache_dtype: Optional[str] = None,
    schedule: Optional[str] = None,
    fp8_qk: bool = False,
) -> Union[torch.Tensor, Tuple[torch.Tensor, torch.Tensor]]:
    """Sparse shared-KV attention forward; returns ``attention_out`` in q's layout.

    With ``return_softmax_lse=True`` returns ``(attention_out, lse)``, lse fp32
    ``[T1, N1]`` (TND) or ``[B, S1, N1]`` (BSND), ``lse = max + ln(sum)`` over
    all attended keys with the sink folded in (api.py:176-184). ``metadata``
    is the output of ``sparse_attn_sharedkv_metadata``; when omitted it is
    built here from the inputs (api.py:335-360). ``schedule="device"`` builds it
    on the GPU instead, so the call never waits for the device (see ``prepare``);
    a ``metadata`` tensor on the GPU is used without being read back.
    ``fp8_qk=True`` (fp8 caches only; no reference counterpart) forms Q·Kᵀ on fp8
    MFMA with each head's query latent quantized to e4m3 (one fp32 scale per
    head); P·V stays bf16. It adds the query's quantization error: within
    atol = rtol = 2e-2 of golden on N(0, 1)-scaled data, not on the reference
    tests' U(-10, 10) data.
    """
    prep = prepare(q, ori_kv=ori_kv, cmp_kv=cmp_kv, cmp_sparse_indices=cmp_sparse_indices,
                   ori_block_table=ori_block_table, cmp_block_table=cmp_block_table,
                   cu_seqlens_q=cu_seqlens_q, seqused_q=seqused_q, seqused_kv=seqused_kv,
                   sinks=sinks, metadata=metadata, softmax_scale=softmax_scale,
                   cmp_ratio=cmp_ratio, ori_mask_mode=ori_mask_mode,
                   cmp_mask_mode=cmp_mask_mode, ori_win_left=ori_win_left,
                   ori_win_right=ori_win_right, layout_q=layout_q, layout_kv=layout_kv,
                   core_num=core_num, topk_cmp=topk_cmp, head_dim_v=head_dim_v,
                   kv_cache_dtype=kv_cache_dtype, schedule=schedule, fp8_qk=fp8_qk,
                   _stream_schedule=True)
    launch(prep)
    return finalize(prep, return_softmax_lse)
