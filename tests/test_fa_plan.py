"""CPU checks of how attention_target's launchers pick a form from the sizes."""

import ctypes as ct
import time

import pytest

from ascendflow_amd import _native


def fa_params(b, hq, hkv, causal=False):
    return _native.FaParams(B=b, HQ=hq, HKV=hkv, D=128, dtype=0, causal=int(causal), scale=1.0, reserved=0)


@pytest.mark.parametrize("b,hq,hkv,sq,sk", [(16, 32, 8, 16, 8192), (1, 32, 32, 8192, 8192), (8, 32, 8, 16, 40000)])
def test_the_choice_costs_little_host_time(b, hq, hkv, sq, sk):
    """Every launch makes the choice again, so it must not walk all split
    counts: at most 2.5x a call with nothing to choose from (walking all four
    row tiles' 64 split counts: 4x and more)."""
    lib = _native.library()

    def microseconds(params, sq, sk):
        nbytes = ct.c_uint64(0)
        args = (ct.byref(nbytes), sq, sk, ct.byref(params))
        best = float("inf")
        for _ in range(20):
            start = time.perf_counter()
            for _ in range(300):
                lib.workspace_size_attention_target_split(*args)
            best = min(best, time.perf_counter() - start)
        return best / 300 * 1e6

    assert microseconds(fa_params(b, hq, hkv), sq, sk) < 2.5 * microseconds(fa_params(1, 4, 4), 16, 16)
