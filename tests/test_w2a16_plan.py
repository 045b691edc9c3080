"""What the weight-only entry point decides to launch (slimk_w2a16_gemm_plan), on the host."""
import ctypes
import random

import pytest

from slimkernels_amd import _lib


def plan(M, N, K, g, split_k=0):
    """(token rows of a tile, 0: the few-rows kernel; K splits; K parts inside a workgroup)"""
    out = [ctypes.c_int() for _ in range(3)]
    _lib.check(_lib.lib().slimk_w2a16_gemm_plan(M, N, K, g, split_k, *[ctypes.byref(v) for v in out]))
    return tuple(v.value for v in out)


def no_split_is_empty(K, splits):
    pairs = K // 128
    per = -(-pairs // splits)
    return (splits - 1) * per < pairs


@pytest.mark.parametrize("M,N,K,g,split", [
    (64, 4096, 18688, 128, 0),      # 146 pairs of steps: sixteen splits of ten would leave the last one empty
    (1000, 4096, 257 * 128, 128, 64),  # 257 pairs in 64 splits of five: 52 of them have work
])
def test_rounding_to_pairs_of_steps_leaves_no_split_empty(M, N, K, g, split):
    rows, splits, _ = plan(M, N, K, g, split)
    assert rows > 0 and splits > 1 and no_split_is_empty(K, splits)
    if split:
        assert splits == 52
    else:
        assert splits == _lib.lib().slimk_w2a16_gemm_auto_split_k(M, N, K, g)


def test_no_plan_has_an_empty_split():
    rng = random.Random(11)
    tiled = 0
    for _ in range(4000):
        g = rng.choice([64, 128, 256])
        K = max(g, 128) * rng.randint(1, 40960 // max(g, 128))
        M, N = int(2 ** rng.uniform(0, 12)), int(2 ** rng.uniform(4, 15))
        granules = K // max(g, 128)
        asked = rng.choice([0, 0, rng.randint(1, max(1, min(64, granules // 4)))])
        rows, splits, halves = plan(M, N, K, g, asked)
        assert rows in (0, 64, 128) and halves in (1, 2) and (halves == 1 or rows == 64)
        assert 1 <= splits <= 64 and (splits == 1 or splits * 4 <= granules)
        if asked:
            assert splits <= asked and (rows or splits == asked)
        if rows:
            tiled += 1
            assert no_split_is_empty(K, splits), (M, N, K, g, asked, splits)
            # the launch asks for the plan again with the split it was given: the same split comes out
            assert plan(M, N, K, g, splits)[1] == splits
    assert tiled > 500
