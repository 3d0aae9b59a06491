"""CCOIL_AUTOTUNE against the untuned call: the tuner times the rule's own shape, so that it never replays a slower one."""
import numpy as np
import pytest
import torch

import ccoil_abi as abi
from test_gpu_reduced_rules import _row

pytestmark = pytest.mark.gpu


# a whole wave per point; one lane per point where the visit order costs more than the kernel saves
@pytest.mark.parametrize("coil,n", [(("RECTANGULAR", 0.1, 0.1, 0.1, 59, 27), 4096), (("RECTANGULAR", 0.1, 0.1, 0.1, 59, 27), 300000)])
def test_tuned_call_is_not_slower(coil, n):
    """Device time of the replayed shape within 15 % of the untuned call's, the least of several of either."""
    ctx = abi.Context(0)
    try:
        cs = abi.CoilSet.from_rows([_row(*coil)])
        pts = torch.from_numpy(np.random.default_rng(1).normal(scale=0.2, size=(n, 3))).cuda()
        out = {"B": torch.empty_like(pts)}
        ms = {}
        for flags in (0, abi.AUTOTUNE):
            reps = [ctx.fields(cs, pts, abi.B, abi.FP64, flags | abi.DEVICE_POINTERS, out=out)[1] for _ in range(12)]
            ms[flags] = min(r.kernel_ms for r in reps[2:])
        print(f"\n{n} points: {1e3 * ms[0]:.0f} us, tuned {1e3 * ms[abi.AUTOTUNE]:.0f} ({reps[-1].split} lanes)")
        assert ms[abi.AUTOTUNE] <= 1.15 * ms[0]
    finally:
        ctx.close()
