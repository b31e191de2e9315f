"""Calls of two work items per CU and more at D = 128 and 256: the one-item
kernel serves them and leaves the row-list plan in the workspace. The plan
equals the oracle's selection for every token, and the output equals the
persistent kernel's over that plan bit for bit, either side of the line."""

import pytest
import torch

from oracle import sparse_reference as sr
from tests.sparse_helpers import assert_close, assert_plan_matches, call_args, call_kwargs, guard_intact, to_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("items", [511, 512, 513])
@pytest.mark.parametrize(
    "d,h,bm,topk,case",
    [(128, 32, 32, 512, "ragged"), (256, 32, 32, 300, "padding"), (256, 64, 64, 1024, "mixed"), (128, 64, 64, 7, "empty")],
)
def test_plan_and_output_match_the_persistent_kernel(device, d, h, bm, topk, case, items):
    from ascendflow_amd.sparse_attention import sparse_mla, sparse_mla_planned
    from ascendflow_amd.sparse_attention.attention import workspace_bytes
    from ascendflow_amd.sparse_attention.probe import sparse_mla_plan

    print(f"\n[sparse narrow] D={d} H={h} BM={bm} TOPK={topk} {case} items={items}", flush=True)
    policy = sr.default_policy(B=5, T=items, H=h, D=d, BM=bm, MAX_SEQ=2048, TOPK=topk, ORI_BLOCKS=80, CMP_BLOCKS=80,
                               DTYPE="bf16" if d == 128 else "f16")
    policy["SCALE"] = d ** -0.5
    data = sr.inputs(policy, case)
    tensors = to_device(data, policy, device)
    size_keys = ("B", "T", "H", "D", "PAGE", "RATIO", "MAX_SEQ", "ORI_BLOCKS", "CMP_BLOCKS", "WINDOW", "TOPK", "S",
                 "BM", "DTYPE", "SCALE")
    workspace = torch.full((workspace_bytes(**{k: policy[k] for k in size_keys}, parts=1),), 0xCD, dtype=torch.uint8,
                           device=device)
    lse = torch.full((items, h), float("nan"), dtype=torch.float32, device=device)
    sparse_mla(*call_args(tensors), **call_kwargs(policy), workspace=workspace, parts=1, softmax_lse=lse)
    torch.cuda.synchronize()
    assert guard_intact(tensors), "kernel wrote past attention_out"
    if items >= 512:
        assert_plan_matches(workspace, data, policy, list(range(items)))
    else:
        assert bool((workspace == 0xCD).all()), "below two items per CU the workspace is not written"
    out = tensors["attention_out"].clone()
    sample = [0, 1, items // 2, items - 1]
    assert_close(out.float().cpu().numpy()[sample], sr.oracle_fp32(data, policy, sample), policy["DTYPE"])
    for t in (tensors["attention_out"], lse):
        t.fill_(float("nan"))
    sparse_mla(*call_args(tensors), **call_kwargs(policy), softmax_lse=lse)  # no plan left, perhaps split keys
    torch.cuda.synchronize()
    if items >= 512:
        assert torch.equal(out, tensors["attention_out"])
    else:
        assert_close(tensors["attention_out"].float().cpu().numpy()[sample], sr.oracle_fp32(data, policy, sample),
                     policy["DTYPE"])
    sparse_mla(*call_args(tensors), **call_kwargs(policy), parts=1, softmax_lse=lse)
    planned_lse = torch.empty_like(lse)
    kw = call_kwargs(policy)
    sparse_mla_planned(*(tensors[k] for k in ("q", "ori_kv", "cmp_kv", "sinks", "attention_out")),
                       sparse_mla_plan(tensors, policy), softmax_lse=planned_lse, **kw)
    torch.cuda.synchronize()
    assert torch.equal(out, tensors["attention_out"]) and torch.equal(lse, planned_lse)
