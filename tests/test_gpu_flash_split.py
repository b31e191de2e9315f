"""The split-key flash-attention kernel (packed query rows, one stream of keys
per wave) and its merge, at the edges of its tiles, against the online oracle
at the contract tolerance of test_gpu_flash.py: packed rows either side of each
row tile, keys either side of the 32-key tile, of one tile per wave and of a
split, causal row tiles inside one head and across heads, and the form with
non-temporal loads (128 MiB of KV and more). Every case states the form that the
sizes choose and checks it."""

import ctypes as ct

import numpy as np
import pytest
import torch

from ascendflow_amd import _native
from oracle.attention import inputs
from tests.test_gpu_flash import TORCH, assert_contract, online_rows, run_fa, sampled_rows


def form_of(b, hq, hkv, sq, sk, causal, workspace=True):
    """(kernel: 0 forward, 1 packed rows; query rows per workgroup; key splits) of a call."""
    params = _native.FaParams(B=b, HQ=hq, HKV=hkv, D=128, dtype=0, causal=int(causal), scale=1.0, reserved=0)
    form = (ct.c_int64 * 3)()
    assert _native.library().form_attention_target(form, sq, sk, ct.byref(params), int(workspace)) == 0
    return tuple(form)


@pytest.mark.gpu
@pytest.mark.parametrize(
    "b,hq,hkv,sq,sk,dtype,causal,case,form",
    [
        # Grids of few rows and keys: the forward kernel's 64-row tiles.
        (1, 4, 4, 1, 1, "bf16", False, "standard", (0, 64, 1)),
        (2, 8, 2, 1, 31, "f16", False, "standard", (0, 64, 1)),
        (1, 8, 2, 4, 33, "bf16", False, "sharp", (0, 64, 1)),
        (1, 17, 1, 1, 129, "f16", False, "standard", (0, 64, 1)),
        (1, 3, 1, 11, 127, "bf16", False, "standard", (0, 64, 1)),
        (1, 28, 4, 3, 500, "bf16", True, "standard", (0, 64, 1)),
        (1, 4, 2, 250, 700, "f16", True, "standard", (0, 64, 1)),
        # Whole keys: waves without a tile, tiles either side of 32 keys and of one per wave, 7 to 168 packed rows.
        (19, 28, 4, 1, 1, "bf16", False, "standard", (1, 16, 1)),
        (19, 28, 4, 1, 31, "f16", False, "sharp", (1, 16, 1)),
        (19, 28, 4, 1, 33, "bf16", False, "standard", (1, 16, 1)),
        (20, 28, 4, 2, 127, "f16", False, "standard", (1, 16, 1)),
        (19, 28, 4, 7, 129, "bf16", False, "sharp", (1, 32, 1)),
        (19, 28, 4, 16, 33, "f16", False, "standard", (1, 48, 1)),
        (19, 28, 4, 24, 65, "bf16", False, "standard", (1, 64, 1)),
        (19, 28, 4, 24, 129, "f16", False, "sharp", (1, 64, 1)),
        # Split keys, either side of each row tile.
        (1, 1, 1, 1, 500, "bf16", False, "standard", (1, 16, 4)),
        (1, 17, 1, 1, 1129, "f16", False, "standard", (1, 16, 9)),   # 17 rows: two row tiles
        (1, 3, 1, 11, 2127, "bf16", False, "sharp", (1, 16, 9)),     # 33 rows
        (1, 7, 1, 7, 4097, "f16", False, "sharp", (1, 16, 17)),      # 49 rows
        (2, 8, 2, 16, 4100, "bf16", False, "standard", (1, 32, 17)),  # 64 rows
        (1, 5, 1, 13, 2050, "bf16", False, "standard", (1, 16, 9)),  # 65 rows
        (3, 4, 1, 100, 1000, "f16", False, "standard", (1, 48, 8)),
        (1, 32, 8, 1, 9001, "bf16", False, "sharp", (1, 16, 18)),
        (1, 8, 8, 200, 3000, "f16", False, "standard", (1, 64, 8)),
        (8, 32, 8, 1, 4128, "bf16", False, "standard", (1, 16, 3)),  # 135 MB of KV: non-temporal loads
        # Causal: row tiles across heads, whole heads in one tile and parts of them.
        (19, 32, 8, 2, 2, "bf16", True, "standard", (1, 16, 1)),
        (19, 28, 4, 7, 40, "f16", True, "sharp", (1, 32, 1)),
        (27, 28, 4, 12, 12, "bf16", True, "standard", (1, 48, 1)),
        (12, 64, 8, 11, 100, "f16", True, "standard", (1, 48, 1)),
        (28, 32, 8, 13, 263, "bf16", True, "sharp", (1, 64, 1)),
        # Causal: one head per row tile, split keys, some splits past a tile's last query.
        (1, 1, 1, 512, 700, "f16", True, "standard", (1, 16, 4)),
        (1, 4, 2, 512, 700, "bf16", True, "standard", (1, 32, 4)),
        (3, 1, 1, 640, 700, "f16", True, "sharp", (1, 48, 5)),
        (1, 4, 4, 640, 700, "bf16", True, "standard", (1, 64, 5)),
        (1, 8, 8, 1000, 1000, "bf16", True, "sharp", (1, 32, 1)),
    ],
)
def test_split_kernel_matches_the_reference_contract(device, b, hq, hkv, sq, sk, dtype, causal, case, form):
    print(f"\n[fa split] b={b} hq={hq} hkv={hkv} sq={sq} sk={sk} {dtype} causal={causal} case={case}", flush=True)
    assert form_of(b, hq, hkv, sq, sk, causal) == form, "the call runs another kernel than this case is for"
    data = inputs(b, hq, hkv, sq, sk, dtype, scale=0.5, case=case)
    actual = run_fa(data, dtype, causal, device)
    rows = np.arange(sq) if sq <= 64 else sampled_rows(sq)
    few = sorted({0, 1, b // 2, b - 1} & set(range(b))) if hq > 16 else list(range(b))  # every entry is finite, these are compared
    assert np.isfinite(actual).all()
    expected = online_rows(data["q"][few], data["k"][few], data["v"][few], rows, dtype, causal, 32)
    assert_contract(actual[few][:, :, rows], expected, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_infinite_scores_in_split_keys(device, dtype):
    """Keys of score -inf (one, a whole split, all but one key) weigh nothing,
    wherever the splits end; one key of score +inf makes its rows NaN, as
    softmax does, and no other row."""
    from ascendflow_amd.flash_attention import attention_target

    b, hq, hkv, sk = 4, 4, 1, 4100
    assert form_of(b, hq, hkv, 1, sk, False)[0] == 1 and form_of(b, hq, hkv, 1, sk, False)[2] > 1
    data = inputs(b, hq, hkv, 1, sk, dtype, scale=0.5)
    data["q"][..., 0] = np.abs(data["q"][..., 0]) + 0.5  # so that feature 0 of a key sets its score's sign
    masked = np.zeros((b, sk), bool)
    masked[0, 17] = True
    masked[1, 100:3000] = True
    masked[2, :] = True
    masked[2, 2222] = False
    for i in range(b):
        data["k"][i, 0, masked[i], 0] = -np.inf
    data["k"][3, 0, 4000, 0] = np.inf
    q, k, v = (torch.from_numpy(data[n]).to(device, TORCH[dtype]) for n in ("q", "k", "v"))
    o = torch.full_like(q, 7.0)
    attention_target(q, k, v, o, 1, sk, B=b, HQ=hq, HKV=hkv, D=128, DTYPE=dtype, SCALE=128**-0.5)
    actual = o.float().cpu().numpy()
    for i in range(3):
        keep = ~masked[i]
        expected = online_rows(q[i:i + 1].float().cpu().numpy(), data["k"][i:i + 1][:, :, keep],
                               data["v"][i:i + 1][:, :, keep], np.arange(1), dtype, False, 32)
        assert_contract(actual[i:i + 1], expected, dtype)
    assert np.isnan(actual[3]).all()


def test_split_entry_refuses_a_small_workspace():
    """A call that splits its keys is refused, before any launch, without the workspace it asks for."""
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
