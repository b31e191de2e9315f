"""Teaching attention with one resident 128-row KV tile, on MI355X.

Drop-in for ``examples/flash_attention/simple.py:60-69`` (``simple_attention``):
``softmax(Q K^T / sqrt(128)) V`` per head, FP16 Q/K/V/P/O with FP32 scores,
P normalised before its FP16 cast. Launches ``launch_simple_attention``.
"""

from __future__ import annotations

import torch

from .. import _native
from .._tensors import Operand, kept_by_value, operand_pointers, raw_stream, require


@kept_by_value
def _operands(S, H, GROUPS):
    """Operands of a call of checked sizes."""
    require(S > 0 and S % 64 == 0, "S must be a positive multiple of 64")
    require(H > 0 and GROUPS > 0, "positive head and worker counts")
    return (Operand("Q", (H, S, 128), torch.float16), Operand("K", (H, 128, 128), torch.float16),
            Operand("V", (H, 128, 128), torch.float16), Operand("O", (H, S, 128), torch.float16))


def simple_attention(Q, K, V, O, S=256, H=4, GROUPS=20):
    device, (q, k, v, o) = operand_pointers(_operands(S, H, GROUPS), (Q, K, V, O), 3)
    status = _native.library().launch_simple_attention(raw_stream(device), q, k, v, o, None, S, H)
    if status:
        _native.check(status, "launch_simple_attention")
    return O
