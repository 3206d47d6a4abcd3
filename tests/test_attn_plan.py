"""How attention steps split their keys (attn_plan, attn_flash_plan of the
library), on the CPU: every plan covers the visible keys in splits that each
hold some, and its partials fit the room that is reserved for them at once,
so that no step frees partials that a captured graph writes to."""
import ctypes as C
import re
import subprocess

import numpy as np
import pytest

from overhang_amd import gdn

FLASH_ROOM, SPLIT_ROOM = 128 << 20, 8 << 20       # kFlashPartialBytes, kSplitPartialBytes

# query heads, kv heads, head width
SHAPES = [(16, 2, 256), (8, 2, 128), (16, 1, 128), (4, 4, 256), (64, 8, 128), (32, 8, 64), (30, 2, 64), (8, 8, 32), (16, 1, 32)]


def _function(name):
    out = subprocess.run(["nm", "-D", "--defined-only", gdn.LIB_PATH], capture_output=True, text=True).stdout
    return gdn.lib()[re.search(rf"\b_ZN3omh{len(name)}{name}E\w+", out).group(0)]


def _plan(f, *args):
    ns, kps = C.c_int(), C.c_int()
    f(*args, C.byref(ns), C.byref(kps))
    return ns.value, kps.value


def _steps(rng, lo, hi, n):
    """(pos, T), both spread over their logarithms."""
    T = np.exp(rng.uniform(np.log(lo), np.log(hi + 1), n)).astype(int)
    pos = np.exp(rng.uniform(0, np.log(1 << 18), n)).astype(int) - 1
    return list(zip(pos.tolist(), T.tolist())) + [(0, lo), (0, hi), (1 << 18, lo), (1 << 18, hi)]


@pytest.mark.parametrize("H,KV,hd", SHAPES)
def test_split_plan(H, KV, hd):
    f = _function("attn_plan")
    for pos, T in _steps(np.random.default_rng(3), 1, 63 if hd >= 128 else 4096, 3000):
        ns, kps = _plan(f, pos, T, H, KV, hd)
        assert ns >= 1 and kps % 64 == 0 and (ns - 1) * kps < pos + T <= ns * kps, (pos, T, ns, kps)
        assert ns == 1 or T * H * ns * hd * 4 <= SPLIT_ROOM, (pos, T, ns)


@pytest.mark.parametrize("H,KV,hd", [s for s in SHAPES if s[2] >= 128])
def test_flash_plan(H, KV, hd):
    f = _function("attn_flash_plan")
    for pos, T in _steps(np.random.default_rng(4), 64, 40000, 3000):
        for most in (1 << 40, 3, 1):
            ns, kps = _plan(f, pos, T, H, KV, hd, C.c_long(most))
            assert 1 <= ns <= most and kps % 32 == 0 and (ns - 1) * kps < pos + T <= ns * kps, (pos, T, most, ns, kps)
            assert ns == 1 or T * H * ns * hd * 4 <= FLASH_ROOM, (pos, T, ns)
