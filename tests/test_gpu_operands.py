"""The operand checks of the attention and top-k entries (one pass per call):
each wrong operand is refused with its name before any launch, and a call whose
output overlaps an input is refused."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def call_of(entry, device):
    """(tensors by name in order, call(tensors), index of the output) of a small valid call."""
    if entry == "fa":
        from ascendflow_amd.flash_attention import attention_target

        t = [torch.zeros((1, 2, 16, 128), dtype=torch.bfloat16, device=device) for _ in range(4)]
        return ["Q", "K", "V", "O"], t, lambda x: attention_target(*x, 16, 16, B=1, HQ=2, HKV=2, D=128, DTYPE="bf16"), 3
    if entry == "simple":
        from ascendflow_amd.flash_attention import simple_attention

        t = [torch.zeros((2, 128, 128), dtype=torch.float16, device=device) for _ in range(4)]
        return ["Q", "K", "V", "O"], t, lambda x: simple_attention(*x, S=128, H=2), 3
    from ascendflow_amd.sparse_attention import sparse_topk_indices

    i32 = dict(dtype=torch.int32, device=device)
    t = [torch.zeros((2, 64), device=device), torch.tensor([0, 2], **i32), torch.tensor([64], **i32),
         torch.tensor([0], **i32), torch.empty((2, 1, 8), **i32)]
    names = ["scores", "cu_seqlens_q", "seqused_cmp_kv", "cmp_residual_kv", "cmp_sparse_indices"]
    return names, t, lambda x: sparse_topk_indices(*x[:4], TOPK=8, RATIO=2, out=x[4]), 4


@pytest.mark.parametrize("entry", ["fa", "simple", "topk"])
def test_wrong_operands_are_refused_by_name(device, entry):
    names, tensors, call, output = call_of(entry, device)
    assert call(tensors) is tensors[output]
    for i, name in enumerate(names):
        good = tensors[i]
        wrong = {"dtype": good.double(), "device": good.cpu(), "shape": torch.cat([good, good])}
        if good.dim() > 1:
            wrong["contiguous"] = torch.stack([good, good], dim=-1)[..., 0]
        for what, bad in wrong.items():
            if entry == "topk" and i < 2 and what == "shape":
                continue  # the sizes come from these two: another size is another valid call
            with pytest.raises(ValueError, match=name if i else ".*"):
                call([*tensors[:i], bad, *tensors[i + 1:]])
    if entry == "topk":
        indices_in_scores = tensors[0].view(torch.int32).view(-1)[16:32].view(2, 1, 8)
        cu_in_indices = tensors[4].view(-1)[14:]
        cu_in_indices.copy_(tensors[1])
        overlapping = [tensors[:4] + [indices_in_scores], [tensors[0], cu_in_indices, *tensors[2:]]]
    else:
        overlapping = [[tensors[output], *tensors[1:]], [tensors[0], tensors[output], *tensors[2:]]]
    for operands in overlapping:
        with pytest.raises(ValueError, match="overlap"):
            call(operands)
    torch.cuda.synchronize()
