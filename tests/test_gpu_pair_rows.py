"""Pair batches of more work items or pairs than one row of a launch's blocks (2^22)."""
import numpy as np
import pytest

import ccoil_abi as abi
from test_gpu_reduced_rules import _row

pytestmark = pytest.mark.gpu


def test_items_beyond_a_row(ctx):
    """One pair whose secondary has 1.8e8 blocks of 100 nodes, 4.4 million items (and digits beyond a float quotient's reach): the
    value of 20 blocks, both converged."""
    prim = _row("FILAMENT", 0.25, 0.0, 0.0, 2, 1)
    M = []
    for blocks in (20, 180_000_000):
        s = _row("FILAMENT", 0.1, 0.0, 0.0, 100, 1)
        s.update(pos=(0.1, 0.2, 0.5), alpha=0.4, beta=1.2, n_len=1, blocks=(1, 1, blocks))
        P, S = abi.CoilSet.from_rows([prim]), abi.CoilSet.from_rows([s])
        M.append(ctx.pairs(P, S, 1, abi.PAIR_M, abi.FP64)[0]["M"][0])
    assert abs(M[1] - M[0]) <= 1e-10 * abs(M[0])


def test_pairs_beyond_a_row(ctx):
    prim, s = _row("FILAMENT", 0.25, 0.0, 0.0, 6, 1), _row("FILAMENT", 0.1, 0.0, 0.0, 6, 1)
    s.update(pos=(0.1, 0.2, 0.5), alpha=0.4, beta=1.2, n_len=1)
    P, S, n = abi.CoilSet.from_rows([prim]), abi.CoilSet.from_rows([s]), (1 << 22) + 5
    i = np.zeros(n, dtype=np.int64)
    M = ctx.pairs(P, S, n, abi.PAIR_M, abi.FP64, prim_index=i, sec_index=i)[0]["M"]
    assert np.all(M == M[0]) and abs(M[0] - ctx.pairs(P, S, 1, abi.PAIR_M, abi.FP64)[0]["M"][0]) <= 1e-12 * abs(M[0])
