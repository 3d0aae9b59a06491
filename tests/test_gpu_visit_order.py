"""The visit order of calls with many points (spatial cells, counting sort): its time where points crowd, and its values."""
import numpy as np
import pytest

import ccoil_abi as abi
from test_gpu_reduced_rules import _row

pytestmark = pytest.mark.gpu


def _coils(coil, copies, rng):
    rows = []
    for _ in range(copies):
        row = _row(*coil)
        row.update(pos=tuple(rng.normal(scale=0.3, size=3)), alpha=float(rng.uniform(0, 3)), beta=float(rng.uniform(0, 6)))
        rows.append(row)
    return abi.CoilSet.from_rows(rows)


# 2^18 points. A normal cloud's waves take more classes than a uniform one's, 1.4 times the time with 8 points a cell on
# average; 1.8 and 2.3 times with 64, thousands of them in the middle cells
@pytest.mark.parametrize("nodes,copies", [(48, 24), (100, 6)])
def test_time_of_a_dense_cloud(ctx, nodes, copies):
    n = 1 << 18
    rng = np.random.default_rng(1)
    cs = _coils(("THIN", 0.3, 0.0, 0.2, nodes, 1), copies, rng)
    us = {}
    for name, pts in (("normal", rng.normal(scale=0.4, size=(n, 3))), ("uniform", rng.uniform(-0.8, 0.8, size=(n, 3)))):
        us[name] = 1e3 * min(ctx.fields(cs, pts, abi.B, abi.FP64)[1].kernel_ms for _ in range(7))
    print(f"\n{copies} coils of {nodes} nodes: normal {us['normal']:.0f} us, uniform {us['uniform']:.0f}")
    assert us["normal"] <= 1.6 * us["uniform"]
