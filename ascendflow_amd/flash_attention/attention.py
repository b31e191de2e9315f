"""BNSD flash attention forward on MI355X.

Drop-in for ``examples/flash_attention/attention.py:243-264`` (``attention_target``)
and its host tiling policy ``causal_policy`` (``attention.py:19-26``). The call
launches the gfx950 kernels of ``csrc/flash_attention.hip`` through
``launch_attention_target_split`` on the current stream: one fused kernel, or,
for few query rows and small grids, a kernel over split keys and the merge of
its partial results. The Ascend tiling
constexprs (BQ, BM, BK, CK, VR, GROUPS) are checked against the reference's
asserts (``attention.py:305-318``) and otherwise ignored.
"""

from __future__ import annotations

import ctypes as ct

import torch

from .. import _native
from .._tensors import DTYPES, Operand, kept_by_value, operand_pointers, raw_stream, require, storage_dtype


def causal_policy(sq, sk):
    """Host tiling policy of the reference (``attention.py:19-26``), unchanged."""
    prefix = min(sq, sk)
    if prefix < 2048:
        return {"kv_tile": 256, "vector_rows": 16}
    if prefix < 8192:
        return {"kv_tile": 512, "vector_rows": 16}
    return {"kv_tile": 1024, "vector_rows": 8}


class _Call:
    """Checked sizes of a call: its operands, launcher parameters and workspace bytes (none changes afterwards)."""

    __slots__ = ("Sq", "Sk", "operands", "params", "nbytes", "launch")


@kept_by_value
def _call(lib, Sq, Sk, B, HQ, HKV, D, BQ, BM, BK, CK, VR, GROUPS, dtype, SCALE, causal):
    require(Sq >= 1 and Sk >= 1, "Sq and Sk must be >= 1")
    require(B > 0 and HQ > 0 and HKV > 0, "positive batch and head counts")
    require(HQ % HKV == 0, "query heads must be divisible by KV heads")
    require(VR > 0 and BQ % (2 * VR) == 0, "query tile must cover complete rows on both AIVs")
    require(BM > 0 and BQ % BM == 0 and BQ <= 2 * BM, "query tile must fit the accumulator planes")
    require(CK > 0 and BK % CK == 0 and CK == D, "KV tile must contain complete CK == D chunks")
    require(GROUPS > 0 and SCALE > 0, "positive worker count and scale")
    require(D == 128, "gfx950 kernel supports D = 128")
    b16 = DTYPES[dtype]
    call = _Call()
    call.Sq, call.Sk = Sq, Sk
    call.operands = (Operand("Q", (B, HQ, Sq, D), b16), Operand("K", (B, HKV, Sk, D), b16),
                     Operand("V", (B, HKV, Sk, D), b16), Operand("O", (B, HQ, Sq, D), b16))
    params = _native.FaParams(
        B=B, HQ=HQ, HKV=HKV, D=D, dtype=_native.AFA_DTYPE[dtype], causal=int(causal), scale=SCALE, reserved=0
    )
    nbytes = ct.c_uint64(0)
    _native.check(lib.workspace_size_attention_target_split(ct.byref(nbytes), Sq, Sk, ct.byref(params)),
                  "workspace_size_attention_target_split")
    call.params = ct.pointer(params)
    call.nbytes = nbytes.value
    call.launch = lib.launch_attention_target_split
    return call


def attention_target(
    Q,
    K,
    V,
    O,
    Sq,
    Sk,
    B=1,
    HQ=8,
    HKV=8,
    D=128,
    BQ=256,
    BM=128,
    BK=1024,
    CK=128,
    VR=8,
    GROUPS=20,
    DTYPE="f16",
    SCALE=0.08838834764831845,
    CAUSAL=False,
):
    """FA forward: O[B,HQ,Sq,D] = softmax(Q K^T * SCALE [+ causal mask]) V."""
    call = _call(_native.library(), int(Sq), int(Sk), B, HQ, HKV, D, BQ, BM, BK, CK, VR, GROUPS,
                 storage_dtype(DTYPE), SCALE, bool(CAUSAL))
    device, (q, k, v, o) = operand_pointers(call.operands, (Q, K, V, O), 3)
    workspace = None
    if call.nbytes:
        # Partial results of split keys; the caching allocator keeps the block for this stream.
        scratch = torch.empty(call.nbytes, dtype=torch.uint8, device=Q.device)
        workspace = scratch.data_ptr()
    status = call.launch(raw_stream(device), q, k, v, o, workspace, call.nbytes, call.Sq, call.Sk, call.params)
    if status:
        _native.check(status, "launch_attention_target_split")
    return O
