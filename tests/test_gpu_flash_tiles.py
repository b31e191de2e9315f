"""The forward flash-attention kernel in tiles of 128 and 64 query rows (four
waves, two slots per tensor in the KV ring): one, two and more key chunks, a
ragged last one, tiles either side of their rows, causal and grouped heads,
against the online oracle at the contract tolerance of test_gpu_flash.py; and
causal calls whose keys fit the Infinity Cache (tiles of all heads by length)
and do not (tiles head by head)."""

import numpy as np
import pytest
import torch

from oracle.attention import inputs
from tests.test_gpu_flash import TORCH, assert_contract, online_rows, run_fa
from tests.test_gpu_flash_split import form_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "b,hq,hkv,sq,sk,dtype,causal,case,tile",
    [
        # 64-row tiles: small grids, and short keys on large ones
        (1, 8, 8, 64, 1, "f16", False, "standard", 64),
        (2, 8, 2, 65, 64, "bf16", False, "standard", 64),
        (2, 8, 2, 129, 65, "f16", False, "sharp", 64),
        (1, 2, 2, 63, 191, "bf16", True, "standard", 64),
        (1, 4, 1, 700, 300, "bf16", True, "sharp", 64),
        (2, 8, 2, 300, 300, "f16", True, "standard", 64),
        (48, 8, 8, 257, 64, "bf16", True, "standard", 64),
        (40, 16, 16, 129, 65, "f16", False, "standard", 64),
        (40, 16, 4, 127, 128, "bf16", False, "sharp", 64),
        (64, 8, 8, 129, 129, "bf16", True, "standard", 64),
        # 128-row tiles
        (48, 8, 8, 120, 193, "f16", False, "standard", 128),
        (40, 16, 4, 127, 256, "bf16", False, "sharp", 128),
        (64, 8, 8, 129, 193, "f16", False, "standard", 128),
        (48, 8, 8, 257, 257, "bf16", True, "standard", 128),
        (12, 32, 32, 257, 300, "f16", True, "sharp", 128),
    ],
)
def test_tiles_match_the_reference_contract(device, b, hq, hkv, sq, sk, dtype, causal, case, tile):
    print(f"\n[fa tiles] b={b} hq={hq} hkv={hkv} sq={sq} sk={sk} {dtype} causal={causal} case={case}", flush=True)
    assert form_of(b, hq, hkv, sq, sk, causal) == (0, tile, 1)
    data = inputs(b, hq, hkv, sq, sk, dtype, scale=0.5, case=case)
    actual = run_fa(data, dtype, causal, device)
    rows = np.array(sorted({min(r, sq - 1) for r in (0, 15, 16, 62, 63, 64, 127, 128, sq // 2, sq - 1)}))
    few = [0, b // 2, b - 1] if b > 3 else list(range(b))  # every batch entry is finite, these are compared
    assert np.isfinite(actual).all()
    expected = online_rows(data["q"][few], data["k"][few], data["v"][few], rows, dtype, causal, 64)
    assert_contract(actual[few][:, :, rows], expected, dtype)


@pytest.mark.parametrize("b,hq,hkv,sq,sk,dtype", [
    (60, 64, 64, 128, 200, "bf16"),  # 240 MiB of visible keys and values: by length
    (60, 64, 64, 129, 129, "f16"),   # 242 MiB, heads a multiple of the 8 XCDs: head by head
    (75, 27, 27, 257, 300, "bf16"),  # 254 MiB, heads not
])
def test_causal_tile_orders(device, b, hq, hkv, sq, sk, dtype):
    from ascendflow_amd.flash_attention import attention_target

    print(f"\n[fa order] b={b} hq={hq} hkv={hkv} sq={sq} sk={sk} {dtype}", flush=True)
    assert form_of(b, hq, hkv, sq, sk, True)[0] == 0
    torch.manual_seed(sq)
    q, k, v = (torch.randn((b, h, s, 128), device=device, dtype=TORCH[dtype]) * 0.5
               for h, s in ((hq, sq), (hkv, sk), (hkv, sk)))
    o = torch.full_like(q, float("nan"))
    attention_target(q, k, v, o, sq, sk, B=b, HQ=hq, HKV=hkv, D=128, DTYPE=dtype, SCALE=128**-0.5, CAUSAL=True)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(o).all())
    batches, heads = [0, b // 2, b - 1], [0, 1, hq // 2, hq - 1]
    pick = lambda t: t[batches][:, heads].float().cpu().numpy()
    rows = np.array(sorted({0, 63, 64, 127, sq - 2, sq - 1}))
    expected = online_rows(pick(q), pick(k), pick(v), rows, dtype, True, 64)
    assert_contract(pick(o)[:, :, rows], expected, dtype)
