"""Top-k rows whose candidates are a part of the allocated columns (requests of
unequal contexts, a buffer of the largest size): bit-exact against the oracle in
every form that stops at the candidates, TOPK either side of the register form's
two entry buffers at candidate counts up to and past four times it, split rows
whose tokens end inside, at the end of and past the first segment; and a call's
time follows its candidates, not the buffer's columns."""

import numpy as np
import pytest
import torch

from oracle import topk_reference as tr
from tests.test_gpu_topk_rows import scores_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["normal", "ties", "special"])
@pytest.mark.parametrize(
    "c,topk,tokens,contexts",
    [
        (4099, 512, 40, (2047, 2048, 2049, 600, 4099, 1)),         # 1024 threads, loads before the request
        (16000, 1024, 30, (4096, 4097, 1024, 1025, 16000, 9000)),
        (30011, 512, 30, (2048, 4095, 4096, 4097, 30011, 513)),    # 1024 threads, loads after it
        (30011, 1024, 30, (4096, 4200, 8192, 30000, 1025, 0)),
        (8000, 512, 52, (2048, 2049, 512, 513, 8000, 4000)),       # 512 threads
        (16384, 700, 52, (2800, 4096, 4097, 701, 16384, 2047)),
        (30000, 512, 52, (2047, 2049, 8191, 8193, 30000, 14000)),
        (131072, 512, 8, (16383, 16384, 16385, 400, 131072, 40000)),  # split rows
        (140001, 1024, 8, (16384, 18000, 32769, 1030, 140001, 70000)),
        (262145, 512, 12, (16384, 16400, 262145, 3, 100000, 49152)),
    ],
)
def test_selection_stops_at_the_candidates(device, c, topk, tokens, contexts, kind):
    from ascendflow_amd.sparse_attention import sparse_topk_indices

    print(f"\n[topk candidates] C={c} TOPK={topk} T={tokens * len(contexts)} {kind}", flush=True)
    rng = np.random.default_rng(c + topk)
    t = tokens * len(contexts)
    cu = np.arange(0, t + 1, tokens).astype(np.int32)
    seq_cmp = np.array(contexts, np.int32)
    residual = np.full(len(contexts), tokens // 2, np.int32)  # tokens either side of each count
    scores = scores_of(kind, rng, t, c)
    to = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=device)
    buffer = torch.full((t * topk + 64,), 7, dtype=torch.int32, device=device)
    out = buffer[: t * topk].view(t, 1, topk)
    sparse_topk_indices(to(scores), to(cu), to(seq_cmp), to(residual), TOPK=topk, RATIO=1, out=out)
    torch.cuda.synchronize()
    assert torch.all(buffer[t * topk:] == 7), "write past the output"
    np.testing.assert_array_equal(out.cpu().numpy(), tr.topk_indices(scores, cu, seq_cmp, residual, topk, 1))


@pytest.mark.parametrize("t,c", [(512, 30000), (1024, 16000), (1024, 30000), (4000, 16384), (16, 131072)])
def test_time_follows_the_candidates(device, t, c):
    """With an eighth of the columns as candidates a call takes well below the
    full row's time (0.4 to 0.72 of it; 0.85 and more when the whole row is read)."""
    from ascendflow_amd.sparse_attention import sparse_topk_indices

    i32 = dict(dtype=torch.int32, device=device)
    scores = [torch.randn((t, c), device=device) for _ in range(2)]
    requests = min(t, 16)
    cu = torch.tensor([t * i // requests for i in range(requests + 1)], **i32)
    out = torch.empty((t, 1, 512), **i32)

    def microseconds(context):
        meta = cu, torch.full((requests,), context, **i32), torch.zeros((requests,), **i32)
        graph = torch.cuda.CUDAGraph()
        for s in scores:
            sparse_topk_indices(s, *meta, TOPK=512, RATIO=1, out=out)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            for _ in range(5):
                for s in scores:
                    sparse_topk_indices(s, *meta, TOPK=512, RATIO=1, out=out)
        best = float("inf")
        for _ in range(5):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record()
            graph.replay()
            end.record()
            torch.cuda.synchronize()
            best = min(best, begin.elapsed_time(end) * 100)
        return best

    full, short = microseconds(c), microseconds(c // 8)
    print(f"\n[topk candidates] T={t} C={c}: full {full:.1f} us, an eighth {short:.1f} us", flush=True)
    assert short < 0.8 * full
