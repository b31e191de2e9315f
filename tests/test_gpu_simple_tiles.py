"""The single-tile attention where a workgroup walks several tiles of a head:
heads whose tiles do not divide evenly over the workgroups, one tile, and more
tiles than one round of the GPU, against the FP32 reference on every row."""

import numpy as np
import pytest
import torch

from oracle.attention import simple_reference
from oracle.dtypes import rounded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,s", [(1, 64), (3, 192), (37, 1088), (9, 7360), (1, 65600)])
def test_every_row_matches_fp32(device, h, s):
    from ascendflow_amd.flash_attention import simple_attention

    print(f"\n[simple] H={h} S={s}", flush=True)
    rng = np.random.default_rng(h * 1000 + s)
    q, k, v = (rounded(rng.standard_normal((h, rows, 128)).astype(np.float32), "f16") for rows in (s, 128, 128))
    tq, tk, tv = (torch.from_numpy(x).to(device, torch.float16) for x in (q, k, v))
    guarded = torch.full((tq.numel() + 256,), float("nan"), dtype=torch.float16, device=device)
    o = guarded[: tq.numel()].view(tq.shape)
    simple_attention(tq, tk, tv, o, S=s, H=h)
    torch.cuda.synchronize()
    assert torch.isnan(guarded[tq.numel():].float()).all(), "kernel wrote past O"
    # The tolerance of test_gpu_flash.py's full-size case.
    np.testing.assert_allclose(o.float().cpu().numpy(), simple_reference(q, k, v), rtol=0.002, atol=0.0005)
