"""hattn_hstate_plan (the native cascade plan) against HState.plan_cascade on the
CPU: the same cascades and counts, and the same token at which it stops."""
import ctypes
import random

import pytest
import torch

from hattention import _lib
from hattention.base import HStruct, HType
from hattention.recurrent import HState


def _native(counts, htype, n):
    L = len(counts)
    c, out = (ctypes.c_int * L)(*counts), (ctypes.c_ubyte * max(1, n))()
    done = _lib.load().hattn_hstate_plan(c, L, htype.value, n, out)
    return list(out[:done]), list(c)


def _python(counts, htype, n):
    S = HState(2, htype, HStruct.MAMBA2, (1, 1, 1, 1, len(counts)), torch.float32, "cpu")
    S.host_counts = list(counts)
    out = []
    for _ in range(n):
        try:
            out.append(S.plan_cascade())
        except (IndexError, ValueError):
            break
    return out, S.host_counts


@pytest.mark.parametrize("htype", [HType.WEAK, HType.STRONG])
@pytest.mark.parametrize("L", [1, 2, 3, 7, 9])
def test_plan_from_empty(L, htype):
    n = min(2 ** L + 5, 255)
    assert _native([0] * L, htype, n) == _python([0] * L, htype, n)


@pytest.mark.parametrize("htype", [HType.WEAK, HType.STRONG])
def test_plan_from_any_counts(htype):
    rng = random.Random(5)
    for _ in range(200):
        L = rng.randint(1, 32)
        counts = [rng.choice([0, 0, 1 << max(0, e - 1), 1 << e, rng.randint(0, 1 << e)]) if e < 30 else 0
                  for e in range(L)]
        assert _native(counts, htype, 20) == _python(counts, htype, 20), counts
