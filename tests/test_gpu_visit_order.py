"""The visit order of calls with many points (spatial cells, counting sort): its time where points crowd, and its values."""
import numpy as np
import pytest
import torch

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


def test_pieces():
    """More points than one order serves (2^24 at a time): the same bits as in a call of the last of them alone, by calls and
    by a plan, and no more memory kept than an order of 2^24 points takes: 2 x 4 bytes each,
    2 x 8 for each of 2^21 cells, and a quarter to grow."""
    tail = 300001
    n = (1 << 25) + tail
    row = _row("RECTANGULAR", 0.1, 0.1, 0.1, 59, 27)
    cs = abi.CoilSet.from_rows([row])
    pts = torch.rand((n, 3), dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(5))
    pts.mul_(1.6).sub_(0.8)
    out = {"B": torch.empty((n, 3), dtype=torch.float64, device="cuda")}
    mid = slice((1 << 24) - tail // 2, (1 << 24) - tail // 2 + tail)   # across the first edge
    last, inner = pts[-tail:].clone(), pts[mid].clone()
    ctx = abi.Context(0)
    some = {"B": torch.empty((tail, 3), dtype=torch.float64, device="cuda")}
    torch.cuda.synchronize()
    _, rep = ctx.fields(cs, last, abi.B, abi.FP64, abi.DEVICE_POINTERS, out=some)
    assert rep.split == 1
    free = torch.cuda.mem_get_info()[0]
    _, rep = ctx.fields(cs, pts, abi.B, abi.FP64, abi.DEVICE_POINTERS, out=out)
    kept = free - torch.cuda.mem_get_info()[0]
    print(f"\n{n} points: {rep.kernel_ms:.1f} ms, main {rep.main_kernel_ms:.1f}, {kept / 2**20:.0f} MiB kept")
    assert rep.split == 1 and 0 < rep.main_kernel_ms <= rep.kernel_ms
    assert torch.equal(out["B"][-tail:], some["B"])
    ctx.fields(cs, inner, abi.B, abi.FP64, abi.DEVICE_POINTERS, out=some)
    assert torch.equal(out["B"][mid], some["B"])
    assert kept <= 1.25 * (8 * 2**24 + 16 * 2**21) + 2**23   # and the driver's rounding
    eager = out["B"].clone()
    plan = ctx.fields_plan(cs, pts, abi.B, abi.FP64, out)
    for _ in range(2):
        out["B"].zero_()
        torch.cuda.synchronize()
        plan.launch()
        plan.synchronize()
        assert torch.equal(out["B"], eager)
    plan.close()
    ctx.close()
