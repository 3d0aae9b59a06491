"""FP32C pairs whose primary keeps its own rule (no reduced rule has fewer nodes, or the gradient's few angular nodes): their
FP64 nodes go through a queue of their own, in full waves and in what is left at the end.

A secondary wound inside the primary's winding has FP64 nodes only, so FP32C equals FP64 up to the order of the sums (1e-10,
the node terms exceeding the sum a thousand times at most); one that crosses the winding has both kinds (3e-5 of the value
of its pose's neighbourhood, the float nodes' rounding)."""
import numpy as np
import pytest

import ccoil_abi as abi
from test_gpu_reduced_rules import _row

pytestmark = pytest.mark.gpu


# red_x never, red_x from 16 nodes (the gradient: its own), and a primary that has reduced rules beside them
@pytest.mark.parametrize("n_ang,n_thk", [(6, 4), (5, 1), (16, 16), (28, 9), (40, 10)])
# secondary nodes per pair: fewer than a queue pass, a few passes and a remainder, and many
@pytest.mark.parametrize("sec", [(5, 1, 1), (9, 3, 5), (30, 5, 6)])
@pytest.mark.parametrize("copies", [1, 40])
def test_nodes_of_the_own_rule(ctx, n_ang, n_thk, sec, copies):
    prim = _row("RECTANGULAR", 0.1, 0.1, 0.1, n_ang, n_thk)
    prim.update(pos=(0.0, 0.0, 0.0), alpha=0.0, beta=0.0)
    inside = _row("RECTANGULAR", 0.13, 0.03, 0.04, sec[0], sec[1])
    inside.update(pos=(0.0, 0.0, 0.011), alpha=0.0, beta=0.0, n_len=sec[2])
    across = _row("RECTANGULAR", 0.06, 0.02, 0.05, sec[0], sec[1])
    across.update(pos=(0.16, 0.03, 0.02), alpha=0.7, beta=0.4, n_len=sec[2])
    P, S = abi.CoilSet.from_rows([prim] * copies), abi.CoilSet.from_rows([inside, across])
    n = 2 * copies
    pi, si = np.repeat(np.arange(copies), 2), np.tile([0, 1], copies)
    what = abi.PAIR_M | abi.PAIR_FT | abi.PAIR_DM
    ref, _ = ctx.pairs(P, S, n, what, abi.FP64, prim_index=pi, sec_index=si)
    got, _ = ctx.pairs(P, S, n, what, abi.FP32C, prim_index=pi, sec_index=si)
    Mr, Gr, _ = ctx.pairs_grad(P, S, n, abi.FP64, prim_index=pi, sec_index=si)
    Mg, Gg, _ = ctx.pairs_grad(P, S, n, abi.FP32C, prim_index=pi, sec_index=si)
    norm = np.linalg.norm
    m = np.abs(ref["M"][0])
    for k in range(n):
        tol = 1e-10 if k % 2 == 0 else 3e-5
        assert abs(got["M"][k] - ref["M"][k]) <= tol * m and abs(Mg[k] - Mr[k]) <= tol * m, k
        assert norm(got["dM"][k] - ref["dM"][k]) <= tol * m / 0.1, k
        assert norm(got["F"][k] - ref["F"][k]) <= tol * max(norm(ref["F"][k]), norm(ref["F"][1])), k
        assert norm(got["T"][k] - ref["T"][k]) <= tol * max(norm(ref["T"][k]), norm(ref["T"][1])), k
        assert norm(Gg[k] - Gr[k]) <= (tol if k % 2 == 0 else 1e-4) * norm(Gr[k]), k
