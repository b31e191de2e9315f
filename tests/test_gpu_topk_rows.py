"""The register form of the top-k selection (sparse_topk_row) and its split form,
bit-exact against the oracle at the edges of their sizes: rows either side of
each register size, both workgroup sizes, TOPK up to and past what these forms
take, segment edges, calls of more tokens than one pair of launches; the filter
form (its linear histograms and their radix fallback) and the streaming one, also
without a workspace. Every case states the form that the sizes choose and checks
it. Scores: normal, heavy ties, constant, infinities and NaN, masked with -inf,
one outlier that spans the histogram."""

import ctypes as ct

import numpy as np
import pytest
import torch

from ascendflow_amd import _native
from ascendflow_amd._tensors import stream_handle
from ascendflow_amd.sparse_attention.indexer import SparseTopkParams
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


ROW, SPLIT, FILTER, STREAM = range(4)


def form_of(t, c, topk, ratio=1, workspace=True):
    """(form, threads or segments, positions per thread or tokens per pair of launches) of a call."""
    params = SparseTopkParams(3, t, topk, ratio, c)
    form = (ct.c_int64 * 3)()
    assert _native.library().form_sparse_topk_indices(form, ct.byref(params), int(workspace)) == 0
    return tuple(form)


def check(device, t, c, topk, kind, form, ratio=1, short=True, seed=0, workspace=True):
    from ascendflow_amd.sparse_attention import sparse_topk_indices

    print(f"\n[topk rows] T={t} C={c} TOPK={topk} {kind} R={ratio} form={form}", flush=True)
    assert form_of(t, c, topk, ratio, workspace)[:len(form)] == form, "the call runs another form than this case is for"
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
    tensors = [to(a) for a in (scores, cu, seq_cmp, residual)]
    if workspace:
        sparse_topk_indices(*tensors, TOPK=topk, RATIO=ratio, out=out)
    else:
        status = _native.library().launch_sparse_topk_indices(
            stream_handle(device), *(x.data_ptr() for x in tensors), out.data_ptr(),
            ct.byref(SparseTopkParams(3, t, topk, ratio, c)))
        assert status == 0
    torch.cuda.synchronize()
    assert torch.all(buffer[t * topk:] == 7), "write past the output"
    np.testing.assert_array_equal(out.cpu().numpy(), tr.topk_indices(scores, cu, seq_cmp, residual, topk, ratio))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["normal", "ties", "constant", "special", "masked", "lowest", "outlier", "tiny"])
@pytest.mark.parametrize(
    "t,c,topk,form",
    [(3, 4096, 512, (ROW, 1024, 4)), (3, 8193, 512, (ROW, 1024, 16)), (258, 700, 96, (ROW, 512, 8)),
     (4, 70001, 512, (FILTER,)), (4, 90001, 512, (SPLIT, 6)), (2049, 1501, 96, (FILTER,))],
)
def test_score_distributions(device, t, c, topk, kind, form):
    check(device, t, c, topk, kind, form, ratio=2)


@pytest.mark.gpu
@pytest.mark.parametrize(
    "t,c,topk,form",
    [(2, 1, 1, (ROW, 1024, 4)), (2, 63, 64, (ROW, 1024, 4)), (3, 1500, 1408, (ROW, 1024, 4)), (3, 2047, 2046, (FILTER,)),
     (3, 2048, 2040, (FILTER,)), (3, 2049, 400, (ROW, 1024, 4)), (3, 4095, 700, (ROW, 1024, 4)),
     (3, 4097, 768, (ROW, 1024, 8)), (2, 8192, 1024, (ROW, 1024, 8)), (2, 16383, 1408, (ROW, 1024, 16)),
     (2, 16383, 1500, (FILTER,)), (2, 16384, 1, (ROW, 1024, 16)), (2, 16385, 512, (ROW, 1024, 32)),
     (2, 32768, 1408, (ROW, 1024, 32)), (2, 32768, 1536, (FILTER,)), (2, 32769, 512, (FILTER,)),
     (256, 4097, 300, (ROW, 1024, 8)), (257, 4096, 300, (ROW, 512, 8)), (257, 4099, 512, (ROW, 512, 16)),
     (258, 8191, 512, (ROW, 512, 16)), (257, 8193, 1408, (ROW, 512, 32)), (259, 16385, 512, (ROW, 512, 64)),
     (1024, 300, 96, (ROW, 512, 8)), (1025, 300, 96, (FILTER,)), (2049, 300, 96, (FILTER,)), (2049, 301, 96, (FILTER,)),
     (1024, 17000, 512, (ROW, 512, 64)), (1030, 17000, 512, (FILTER,))],
)
def test_row_sizes(device, t, c, topk, form):
    check(device, t, c, topk, "normal", form, ratio=1 + c % 2)


@pytest.mark.gpu
@pytest.mark.parametrize(
    "t,c,topk,kind,form",
    [(2, 65537, 512, "normal", (FILTER,)), (2, 81920, 1, "normal", (FILTER,)), (2, 81921, 1, "normal", (SPLIT, 6)),
     (3, 98303, 1024, "ties", (SPLIT, 6)), (3, 98305, 1408, "special", (SPLIT, 7)), (2, 131073, 2047, "special", (FILTER,)),
     (1, 163840, 3000, "normal", (FILTER,)), (3, 262144, 1408, "normal", (SPLIT, 16)), (2, 262145, 512, "ties", (SPLIT, 17)),
     (2, 262145, 1924, "normal", (SPLIT, 17)), (1, 300003, 1700, "normal", (SPLIT, 19)),
     (1, 524289, 512, "outlier", (SPLIT, 33)), (2, 65600, 16384, "normal", (FILTER,))],
)
def test_split_rows(device, t, c, topk, kind, form):
    check(device, t, c, topk, kind, form, ratio=2)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["normal", "ties", "special"])
def test_split_rows_in_several_pairs_of_launches(device, kind):
    """One token more than a pair of launches has workspace for."""
    form = form_of(260, 262145, 1900)
    assert form == (SPLIT, 17, 259)
    check(device, 260, 262145, 1900, kind, form)


@pytest.mark.gpu
@pytest.mark.parametrize(
    "t,c,topk,kind,form,workspace",
    [(2, 262145, 1925, "normal", (STREAM,), True),  # more entries than the merge takes
     (3, 262145, 512, "special", (STREAM,), False), (2, 300001, 700, "ties", (STREAM,), False),
     (1, 524289, 512, "outlier", (STREAM,), False), (3, 262144, 512, "normal", (FILTER,), False),
     (3, 262144, 1024, "ties", (FILTER,), False), (3, 200001, 512, "special", (FILTER,), False)],
)
def test_rows_that_are_not_split(device, t, c, topk, kind, form, workspace):
    """The streaming form, and the filter form up to its 256K positions: the
    entry without a workspace, and TOPK beyond the merge's."""
    check(device, t, c, topk, kind, form, ratio=2, workspace=workspace)


def test_split_entry_refuses_a_small_workspace():
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
