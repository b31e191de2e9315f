"""CPU checks of what the attention and top-k entries keep per set of sizes:
kept by value of plain numbers alone. A number-like whose value changes between
calls (a tensor, a NumPy array) is read again on each, one without a hash is
accepted, and a float where a count is due is refused, whatever was called before."""

import numpy as np
import pytest
import torch

from ascendflow_amd import _native
from ascendflow_amd.flash_attention import attention, simple
from ascendflow_amd.sparse_attention import indexer


def fa(B=1, SCALE=0.25):
    return attention._call(_native.library(), 16, 16, B, 4, 4, 128, 128, 64, 1024, 128, 8, 20, "bf16", SCALE, False)


def topk(TOPK=8):
    return indexer._call(_native.library(), 4, 100, 1, TOPK, 2)


def test_plain_sizes_are_kept():
    assert fa() is fa() and topk() is topk() and simple._operands(64, 2, 20) is simple._operands(64, 2, 20)


@pytest.mark.parametrize("make", [lambda v: torch.tensor(v), lambda v: np.array(v)])
def test_a_changed_value_is_read_again(make):
    scale, size, k = make(0.25), make(64), make(8)
    assert fa(SCALE=scale).params.contents.scale == 0.25
    assert simple._operands(size, 2, 20)[0].shape == (2, 64, 128)
    assert topk(k).operands[4].shape == (4, 1, 8)
    scale[...], size[...], k[...] = 0.5, 128, 16
    assert fa(SCALE=scale).params.contents.scale == 0.5
    assert simple._operands(size, 2, 20)[0].shape == (2, 128, 128)
    assert topk(k).operands[4].shape == (4, 1, 16) and topk(k).params.contents.TOPK == 16


def test_a_float_count_is_refused_after_the_same_whole_number():
    fa(B=1), topk(TOPK=8), simple._operands(64, 2, 20)
    for call in (lambda: fa(B=1.0), lambda: topk(TOPK=8.0), lambda: simple._operands(64.0, 2, 20)):
        with pytest.raises(TypeError):
            call()
