"""What the weight-only entry point decides to launch (slimk_w2a16_gemm_plan), on the host."""
import ctypes
import random

import pytest

from slimkernels_amd import _lib


def plan(M, N, K, g, split_k=0, workspace=1 << 62):
    """(token rows of a tile, 0: the few-rows kernel; K splits; K parts inside a workgroup)"""
    out = [ctypes.c_int() for _ in range(3)]
    _lib.check(_lib.lib().slimk_w2a16_gemm_plan(M, N, K, g, split_k, workspace, *[ctypes.byref(v) for v in out]))
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


def test_a_call_without_workspace_is_taken_where_the_few_rows_rule_takes_none():
    """The library's own choice of a split must fit the workspace at hand: prompts that ran unsplit with NULL still do."""
    L = _lib.lib()
    for M, N, K in ((300, 14336, 4096), (300, 4096, 14336), (436, 14336, 12288)):
        need = L.slimk_w2a16_gemm_workspace_bytes(M, N, K, 128, 0)
        assert need > 0 and plan(M, N, K, 128)[1] * M * N * 4 == need
        for short in (0, need - 1):
            assert plan(M, N, K, 128, 0, short) == plan(M, N, K, 128, 1)
        assert plan(M, N, K, 128, 0, need) == plan(M, N, K, 128)
    # (explicit requests are not changed, and a few rows still ask for what they need)
    assert plan(300, 14336, 4096, 128, 2, 0)[1] == 2
    assert plan(1, 4096, 14336, 128, 0, 0) == plan(1, 4096, 14336, 128) and plan(1, 4096, 14336, 128)[1] > 1
