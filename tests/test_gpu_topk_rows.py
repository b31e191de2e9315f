"""The register form of the top-k selection (sparse_topk_row) and its split form,
bit-exact against the oracle at the edges of their sizes: rows either side of
each register size, both workgroup sizes, TOPK either side of the entries the
kernel holds, segment edges; and calls of many tokens, which the streaming
form serves (its linear histograms and their radix fallback). Scores: normal, heavy ties, constant, infinities and NaN, masked
with -inf, one outlier that spans the histogram."""

import ctypes as ct

import numpy as np
import pytest
import torch

from oracle import topk_reference as tr


def scores_of(kind, rng, t, c):
    if kind == "ties":
        return rng.integers(-2, 3, (t, c)).astype(np.float32)
    if kind == "constant":
        return np.full((t, c), -1.5, np.float32)
    s = rng.standard_normal((t, c)).astype(np.float32)
    if kind == "special":
        for value, share in ((np.inf, 0.01), (-np.inf, 0.2), (np.nan, 0.01), (-0.0, 0.05), (0.0, 0.05)):
            s[rng.random((t, c)) < share] = value
    elif kind == "masked":
        s[:, c // 3:] = -np.inf
    elif kind == "lowest":
        s[:] = np.finfo(np.float32).min
        s[:, ::3] = -np.inf
    elif kind == "outlier":
        s[:, c // 2] = 3.0e38
        s[:, c // 2 + 1:c // 2 + 2] = -3.0e38
    elif kind == "tiny":
        s *= np.float32(1e-40)
    return s


def check(device, t, c, topk, kind, ratio=1, short=True, seed=0):
    from ascendflow_amd.sparse_attention import sparse_topk_indices

    print(f"\n[topk rows] T={t} C={c} TOPK={topk} {kind} R={ratio}", flush=True)
    rng = np.random.default_rng(seed + t * 7 + c)
    scores = scores_of(kind, rng, t, c)
    # Three requests: one over the whole row, one over part of it, one empty.
    cut = (t + 1) // 2
    cu = np.array([0, cut, cut, t], np.int32)
    seq_cmp = np.array([c, c, max(1, (2 * c) // 3) if short else c], np.int32)
    residual = np.full(3, ratio - 1, np.int32)
    to = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=device)
    buffer = torch.full((t * topk + 64,), 7, dtype=torch.int32, device=device)
    out = buffer[: t * topk].view(t, 1, topk)
    sparse_topk_indices(to(scores), to(cu), to(seq_cmp), to(residual), TOPK=topk, RATIO=ratio, out=out)
    torch.cuda.synchronize()
    assert torch.all(buffer[t * topk:] == 7), "write past the output"
    np.testing.assert_array_equal(out.cpu().numpy(), tr.topk_indices(scores, cu, seq_cmp, residual, topk, ratio))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["normal", "ties", "constant", "special", "masked", "lowest", "outlier", "tiny"])
@pytest.mark.parametrize("t,c,topk", [(3, 4096, 512), (3, 8193, 512), (258, 700, 96), (4, 70001, 512), (2049, 1501, 96)])
def test_score_distributions(device, t, c, topk, kind):
    check(device, t, c, topk, kind, ratio=2)


@pytest.mark.gpu
@pytest.mark.parametrize(
    "t,c,topk",
    [(2, 1, 1), (2, 63, 64), (3, 2047, 2046), (3, 2048, 2040), (3, 2049, 400), (3, 4095, 700), (3, 4097, 768),
     (2, 8192, 1024), (2, 16383, 1500), (2, 16384, 1), (2, 16385, 512), (2, 32768, 1536), (257, 4096, 300),
     (257, 4099, 512), (258, 8191, 512), (259, 16385, 512), (2049, 300, 96), (2049, 301, 96), (1030, 17000, 512)],
)
def test_row_sizes(device, t, c, topk):
    check(device, t, c, topk, "normal", ratio=1 + c % 2)


@pytest.mark.gpu
@pytest.mark.parametrize(
    "t,c,topk,kind",
    [(2, 65537, 512, "normal"), (2, 81920, 1, "normal"), (3, 98303, 1024, "ties"), (2, 131073, 2047, "special"),
     (1, 163840, 3000, "normal"), (2, 262145, 512, "ties"), (1, 300003, 1700, "normal"), (1, 524289, 512, "outlier"),
     (2, 65600, 16384, "normal")],
)
def test_split_rows(device, t, c, topk, kind):
    check(device, t, c, topk, kind, ratio=2)


def test_split_entry_refuses_a_small_workspace():
    from ascendflow_amd import _native
    from ascendflow_amd.sparse_attention.indexer import SparseTopkParams

    lib = _native.library()
    need = ct.c_uint64(0)
    params = SparseTopkParams(1, 4, 512, 2, 524288)
    assert lib.workspace_size_sparse_topk_indices_split(ct.byref(need), ct.byref(params)) == 0
    assert need.value == 4 * 32 * 512 * 8
    p = ct.c_void_p(256)
    for workspace, size in ((None, need.value), (p, need.value - 1)):
        assert lib.launch_sparse_topk_indices_split(None, p, p, p, p, p, workspace, size, ct.byref(params)) == -4
    # The workspace of many long rows is bounded: they go in several pairs of launches.
    many = SparseTopkParams(1, 8192, 512, 2, 524288)
    assert lib.workspace_size_sparse_topk_indices_split(ct.byref(need), ct.byref(many)) == 0
    assert 0 < need.value <= 64 << 20
    small = SparseTopkParams(1, 4, 512, 2, 16384)
    assert lib.workspace_size_sparse_topk_indices_split(ct.byref(need), ct.byref(small)) == 0 and need.value == 0
