"""The record pass (near pairs of CCOIL_FP32C, rule pairs of the series modes): its key counts, its padding and its grid.

Values are compared with those of calls below 2^17 points, which sort and sum their records another way; the two differ
by the rounding of FP64 sums, 1e-12 of the field's largest value. Times are the least of several device times, and their
bounds are ratios within one run.
"""
import numpy as np
import pytest
import torch

import ccoil_abi as abi
from test_gpu_reduced_rules import COILS, _row

pytestmark = pytest.mark.gpu

FLAT80 = ("FLAT", 0.1, 0.05, 0.0, 80, 20)
RECT40 = ("RECTANGULAR", 0.1, 0.1, 0.1, 40, 10)
THIN48 = ("THIN", 0.3, 0.0, 0.2, 48, 1)


def _set(kinds, n, rng, spread=0.3):
    rows = []
    for k in range(n):
        row = _row(*kinds[k % len(kinds)])
        row.update(pos=tuple(rng.normal(scale=spread, size=3)), alpha=float(rng.uniform(0, 3)), beta=float(rng.uniform(0, 6)))
        rows.append(row)
    return abi.CoilSet.from_rows(rows)


# keys counted in LDS (up to 10,240: 208 coils of 49 slots) and in memory, and above 2,048 coils two slots instead of 49
@pytest.mark.parametrize("n_coils", [1, 3, 208, 209, 2100])
def test_many_keys(ctx, n_coils):
    rng = np.random.default_rng(31)
    cs = _set(COILS[:8] if n_coils > 1 else [FLAT80], n_coils, rng)
    pts = rng.normal(scale=0.4, size=(131100, 3))
    got, _ = ctx.fields(cs, pts, abi.B, abi.FP32C, abi.DIRECT)
    ref, _ = ctx.fields(cs, pts[:100000], abi.B, abi.FP32C, abi.DIRECT)
    assert np.max(np.abs(got["B"][:100000] - ref["B"])) <= 1e-12 * np.max(np.abs(ref["B"]))


def test_one_coil_bookkeeping(ctx):
    """Counting and placing the records of one coil, whose few keys every wave counts on, takes at most eight times as
    long as its field kernel."""
    cs = abi.CoilSet.from_rows([_row(*THIN48)])
    pts = torch.from_numpy(np.random.default_rng(1).normal(scale=0.4, size=(1 << 20, 3))).cuda()
    out = {"B": torch.empty_like(pts)}
    reps = [ctx.fields(cs, pts, abi.B, abi.FP32C, abi.DIRECT | abi.DEVICE_POINTERS, out=out)[1] for _ in range(7)]
    main = min(r.main_kernel_ms for r in reps)
    rest = min(r.kernel_ms - r.main_kernel_ms - r.record_ms for r in reps)
    print(f"\nfield kernel {1e3 * main:.0f} us, bookkeeping {1e3 * rest:.0f}")
    assert rest <= 8 * main


def test_capacity_beyond_a_launch():
    """2^28 points and two coils: room for 2^29 records, which split over eight lanes would be more than the 2^32 threads
    of a launch. (A context of its own, which gives some 40 GB back.)"""
    ctx = abi.Context(0)
    try:
        cs = _set([("THIN", 0.25, 0.0, 0.05, 6, 1)], 2, np.random.default_rng(2), 0.1)
        n = 1 << 28
        g = torch.Generator(device="cuda").manual_seed(7)
        pts = torch.rand((n, 3), dtype=torch.float64, device="cuda", generator=g) - 0.5
        out = {"B": torch.empty_like(pts)}
        _, rep = ctx.fields(cs, pts, abi.B, abi.FP32C, abi.DIRECT | abi.DEVICE_POINTERS, out=out)
        assert rep.near_pairs > 1 << 20
        some = torch.cat([pts[:20000], pts[-20000:]])
        ref, _ = ctx.fields(cs, some.cpu().numpy(), abi.B, abi.FP32C, abi.DIRECT)
        got = torch.cat([out["B"][:20000], out["B"][-20000:]]).cpu().numpy()
        # each point by itself: a record left out is the coil's whole field there (float nodes by other lanes, 1e-5)
        err, size = np.linalg.norm(got - ref["B"], axis=1), np.linalg.norm(ref["B"], axis=1)
        assert np.all(err <= 1e-5 * size + 1e-6 * np.median(size))
    finally:
        ctx.close()
        torch.cuda.empty_cache()


@pytest.mark.parametrize("coil,mode,flags", [(FLAT80, abi.FP64, abi.FAR_FIELD), (RECT40, abi.FP32C, 0)])
def test_time_where_the_layout_changes(ctx, coil, mode, flags):
    """40 coils in a cloud that meets most classes rarely: 2^17 points, the least whose records are summed by waves of one
    key, take no longer than 1.6 times those of an eighth fewer. (Float records change their lanes there too, one where
    there were eight, so that long rules' are left out.)"""
    rng = np.random.default_rng(1)
    cs = _set([coil], 40, rng)
    pts = torch.from_numpy(rng.uniform(-0.8, 0.8, size=(1 << 17, 3))).cuda()
    out = {"B": torch.empty_like(pts)}
    ms = {}
    for n in (114688, 1 << 17):
        ms[n] = min(ctx.fields(cs, pts[:n], abi.B, mode, flags | abi.DEVICE_POINTERS, out={"B": out["B"][:n]})[1].record_ms
                    for _ in range(7))
    print(f"\n{coil}: " + ", ".join(f"{n} points {1e3 * v:.0f} us" for n, v in ms.items()))
    assert ms[1 << 17] <= 1.6 * ms[114688]
