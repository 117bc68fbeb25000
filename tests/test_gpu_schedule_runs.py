"""The on-device scheduler's fills walk runs of equal items, a budget per lane,
in floats while the total cost is below 2^20 blocks and in 64 bits above, and
record the chosen fill from checkpoints: word-for-word equality with the host
scheduler where those can go wrong -- one run, every item its own run, walks
longer than the checkpoint strides, items over many cores and many items per
core, bisections longer than one round, and totals on both sides of the limit."""

import pytest
import torch

pytestmark = pytest.mark.gpu

HAS_GPU = torch.cuda.is_available()
requires_gpu = pytest.mark.skipif(not HAS_GPU, reason="needs a ROCm GPU")

if HAS_GPU:
    from sparse_attn_sharedkv_amd.metadata import build_metadata, build_metadata_device

CASES = {
    # every item the same; whole items, exactly one per core, and split in two
    "one_run": dict(act_q=[1] * 64, act_kv=[32768] * 64, heads=128, win=-1, scenario=3, topk=2048),
    "one_run_whole": dict(act_q=[300], act_kv=[9000], heads=64, win=127, scenario=1),
    # one item over every core; a long first or last item beside short ones
    "one_item": dict(act_q=[1], act_kv=[140000], heads=16, win=-1, scenario=2),
    "long_last": dict(act_q=[1] * 9, act_kv=[64] * 8 + [130000], heads=64, win=127, scenario=2),
    "long_first": dict(act_q=[1] * 9, act_kv=[130000] + [64] * 8, heads=64, win=127, scenario=2),
    # neighbours always differ: as many runs as items, more than the checkpoints' least stride
    "no_runs": dict(act_q=[1] * 3000, act_kv=[200 + 97 * (i % 2) for i in range(3000)], heads=64,
                    win=-1, scenario=2),
    # many items per core and a bisection of more than one round
    "deep": dict(act_q=[8192], act_kv=[8192], heads=128, win=127, scenario=3, ratio=4, topk=512),
    "empty_items": dict(act_q=[5, 0, 7, 1], act_kv=[3, 9, 0, 700], heads=64, win=-1, scenario=2),
    # totals of 2^20 - 1024, 2^20 and 2^20 + 1024 costs (an item: 1 + 2 + 1021 blocks)
    "below_limit": dict(act_q=[1] * 1023, act_kv=[1021 * 64] * 1023, heads=64, win=-1, scenario=2),
    "at_limit": dict(act_q=[1] * 1024, act_kv=[1021 * 64] * 1024, heads=64, win=-1, scenario=2),
    "above_limit": dict(act_q=[1] * 1025, act_kv=[1021 * 64] * 1025, heads=64, win=-1, scenario=2),
    "above_ragged": dict(act_q=[3] * 700, act_kv=[50000 + 641 * i for i in range(700)], heads=64,
                         win=127, scenario=2),
}


@requires_gpu
@pytest.mark.parametrize("cores", [1, 2, 63, 256, 512])
@pytest.mark.parametrize("name", list(CASES))
def test_runs_equal_host_schedule(name, cores):
    c = dict(CASES[name])
    print(f"[gpu-schedule-runs] {name} cores={cores}", flush=True)
    args = dict(num_heads=c["heads"], ori_win_left=c["win"], scenario=c["scenario"],
                cmp_ratio=c.get("ratio", 1), cmp_topk=c.get("topk", 0), core_num=cores)
    host = build_metadata(act_q=c["act_q"], act_kv=c["act_kv"], **args)
    lens = [torch.tensor(c[k], dtype=torch.int32, device="cuda") for k in ("act_q", "act_kv")]
    for _ in range(2):  # twice: nothing is carried from one build to the next
        dev = build_metadata_device(batch=len(c["act_q"]), act_q=lens[0], act_kv=lens[1], **args)
        assert torch.equal(dev.cpu(), host)
