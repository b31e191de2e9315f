"""The split-key flash-attention kernel (packed query rows, one stream of keys
per wave) and its merge, at the edges of its tiles, against the online oracle
at the contract tolerance of test_gpu_flash.py: packed rows either side of each
row tile, keys either side of the 32-key tile, of one tile per wave and of a
split, causal row tiles inside one head and across heads, and the form with
non-temporal loads (128 MiB of KV and more)."""

import ctypes as ct

import numpy as np
import pytest
import torch

from oracle.attention import inputs
from tests.test_gpu_flash import assert_contract, online_rows, run_fa, sampled_rows


@pytest.mark.gpu
@pytest.mark.parametrize(
    "b,hq,hkv,sq,sk,dtype,causal,case",
    [
        (1, 4, 4, 1, 1, "bf16", False, "standard"),
        (2, 8, 2, 1, 31, "f16", False, "standard"),
        (1, 8, 2, 4, 33, "bf16", False, "sharp"),       # 16 packed rows, two key tiles
        (1, 17, 1, 1, 129, "f16", False, "standard"),   # 17 rows, one key past a tile per wave
        (1, 3, 1, 11, 127, "bf16", False, "standard"),  # 33 rows
        (1, 7, 1, 7, 4097, "f16", False, "sharp"),      # 49 rows, split keys
        (2, 8, 2, 16, 4100, "bf16", False, "standard"),  # 64 rows
        (1, 5, 1, 13, 2050, "bf16", False, "standard"),  # 65 rows: two row tiles
        (1, 32, 8, 1, 9001, "bf16", False, "sharp"),
        (1, 8, 8, 200, 3000, "f16", False, "standard"),
        (1, 28, 4, 3, 500, "bf16", True, "standard"),    # causal, heads inside one row tile
        (1, 4, 2, 250, 700, "f16", True, "standard"),    # causal, row tiles across heads
        (1, 8, 8, 1000, 1000, "bf16", True, "sharp"),    # causal, one head per row tile
        (8, 32, 8, 1, 4128, "bf16", False, "standard"),  # 135 MB of KV
    ],
)
def test_split_kernel_matches_the_reference_contract(device, b, hq, hkv, sq, sk, dtype, causal, case):
    print(f"\n[fa split] b={b} hq={hq} hkv={hkv} sq={sq} sk={sk} {dtype} causal={causal} case={case}", flush=True)
    data = inputs(b, hq, hkv, sq, sk, dtype, scale=0.5, case=case)
    actual = run_fa(data, dtype, causal, device)
    rows = np.arange(sq) if sq <= 64 else sampled_rows(sq)
    expected = online_rows(data["q"], data["k"], data["v"], rows, dtype, causal, 32)
    assert_contract(actual[:, :, rows], expected, dtype)


def test_split_entry_refuses_a_small_workspace():
    """A call that splits its keys is refused, before any launch, without the workspace it asks for."""
    from ascendflow_amd import _native

    lib = _native.library()
    params = _native.FaParams(B=1, HQ=32, HKV=8, D=128, dtype=0, causal=0, scale=1.0, reserved=0)
    need = ct.c_uint64(0)
    assert lib.workspace_size_attention_target_split(ct.byref(need), 1, 16384, ct.byref(params)) == 0
    assert need.value > 0 and need.value % (32 * 130 * 4) == 0  # splits x rows x (128 + 2) floats
    p = ct.c_void_p(256)
    for workspace, size in ((None, need.value), (p, need.value - 1)):
        assert lib.launch_attention_target_split(None, p, p, p, p, workspace, size, 1, 16384, ct.byref(params)) == -4
    assert lib.launch_attention_target_split(None, p, p, None, p, p, need.value, 1, 16384, ct.byref(params)) == -1
    assert lib.launch_attention_target_split(None, p, p, p, p, p, need.value, 0, 16384, ct.byref(params)) == -2
    assert lib.workspace_size_attention_target_split(ct.byref(need), 8192, 8192, ct.byref(params)) == 0
    assert need.value == 0


@pytest.mark.gpu
def test_split_calls_replay_in_a_graph(device):
    """Split flash attention and split top-k rows, whose workspaces come from
    the graph's pool, captured once and replayed on new inputs with eager calls
    between: each replay equals the eager call bit for bit."""
    from ascendflow_amd.flash_attention import attention_target
    from ascendflow_amd.sparse_attention import sparse_topk_indices

    gen = torch.Generator(device=device)
    gen.manual_seed(3)
    q = torch.empty((2, 8, 1, 128), dtype=torch.bfloat16, device=device)
    k, v = (torch.empty((2, 2, 9000, 128), dtype=torch.bfloat16, device=device) for _ in range(2))
    scores = torch.empty((3, 70000), device=device)
    i32 = dict(dtype=torch.int32, device=device)
    meta = (torch.tensor([0, 3], **i32), torch.tensor([70000], **i32), torch.tensor([0], **i32))
    o, indices = torch.empty_like(q), torch.empty((3, 1, 512), **i32)

    def fill():
        for t in (q, k, v, scores):
            t.normal_(generator=gen)

    def calls():
        attention_target(q, k, v, o, 1, 9000, B=2, HQ=8, HKV=2, D=128, DTYPE="bf16", SCALE=128**-0.5)
        sparse_topk_indices(scores, *meta, TOPK=512, RATIO=2, out=indices)

    fill()
    calls()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        calls()
    for _ in range(3):
        fill()
        calls()
        torch.cuda.synchronize()
        expected = o.clone(), indices.clone()
        o.fill_(float("nan"))
        indices.fill_(-7)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, expected[0]) and torch.equal(indices, expected[1])
