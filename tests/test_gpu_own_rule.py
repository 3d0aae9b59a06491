"""CCOIL_FP64's choice between reduced rules and the coils' own nodes (field_rule), at every launch shape.

Values: against CCOIL_FP64_IEEE, which sums the own nodes whatever the call, per point and relative to the coils' own
field, with the tolerances of test_gpu_reduced_rules.py (its points, its reasons; a sum of identical coils scales both).

Times: the choice is there so that no call takes longer than the own nodes with IEEE division and square root, which
cost about twice CCOIL_FP64's arithmetic. The least of several device times, so that a neighbour's load drops out.
"""
import numpy as np
import pytest

import ccoil_abi as abi
from test_gpu_reduced_rules import _points, _row

pytestmark = pytest.mark.gpu

RECT16 = ("RECTANGULAR", 0.1, 0.1, 0.1, 16, 16)
RECT59 = ("RECTANGULAR", 0.1, 0.1, 0.1, 59, 27)
FLAT20 = ("FLAT", 0.1, 0.05, 0.0, 20, 7)
THIN12 = ("THIN", 0.05, 0.0, 0.05, 12, 1)


# own nodes by 16, 4 and 1 lanes per point, chunks of coils among them; reduced rules by one lane in the visit order
@pytest.mark.parametrize("coil,copies,n,split", [(RECT16, 1, 300, 16), (THIN12, 3, 20001, 4), (FLAT20, 9, 40001, 4),
                                                 (RECT16, 2, 70001, 1), (THIN12, 40, 262145, 1), (RECT59, 24, 65537, 1)])
def test_values(ctx, coil, copies, n, split):
    row = _row(*coil)
    pts, r, z = _points(np.random.default_rng(23), row, n)
    cs = abi.CoilSet.from_rows([row] * copies)
    q = abi.A | abi.B | abi.G
    ref, _ = ctx.fields(cs, pts, q, abi.FP64_IEEE)
    got, rep = ctx.fields(cs, pts, q, abi.FP64)
    assert rep.split == split
    R, a, hb = row["R"], row["a"], 0.5 * row["b"] if row["use_fast"] else 0.0
    zd = np.maximum(np.abs(z) - hb, 0.0)
    rho = np.clip(np.hypot(r, zd), R, R + a)
    eta = np.arccosh(1.0 + ((rho - r) ** 2 + zd * zd) / (2.0 * rho * r))
    y = np.hypot(r, z) / np.hypot(R + a, hb)
    b = np.linalg.norm(ref["B"], axis=1)
    for k, near, far in (("A", 1e-11, 2e-14), ("B", 1e-11, 2e-14), ("G", 1e-6, 2e-13)):
        scale = np.linalg.norm(ref[k], axis=1) + (b * R if k == "A" else b / np.maximum(r, 1e-5 * R) if k == "G" else 0.0)
        tol = np.where(eta > 0.1, far * (1.0 + y) ** 2, near)
        assert np.all(np.linalg.norm(got[k] - ref[k], axis=1) <= tol * scale), k


@pytest.mark.parametrize("coil,copies,n", [(RECT16, 40, 40000), (FLAT20, 128, 40000), (THIN12, 1, 1 << 20), (RECT59, 1, 65536)])
def test_no_slower_than_ieee(ctx, coil, copies, n):
    rng = np.random.default_rng(3)
    rows = []
    for _ in range(copies):
        row = _row(*coil)
        row.update(pos=tuple(rng.normal(scale=0.3, size=3)), alpha=float(rng.uniform(0, 3)), beta=float(rng.uniform(0, 6)))
        rows.append(row)
    cs = abi.CoilSet.from_rows(rows)
    pts = rng.normal(scale=0.4, size=(n, 3))
    ms = {p: min(ctx.fields(cs, pts, abi.B, p)[1].kernel_ms for _ in range(7)) for p in (abi.FP64, abi.FP64_IEEE)}
    print(f"\n{coil} {copies} coils {n} points: {1e3 * ms[abi.FP64]:.0f} us, IEEE {1e3 * ms[abi.FP64_IEEE]:.0f}")
    assert ms[abi.FP64] <= ms[abi.FP64_IEEE]


# pairs: batches of short slow rules, just above and below the size from which they sum their own nodes
@pytest.mark.parametrize("n", [110, 125, 2048])
def test_pairs(ctx, n):
    rng = np.random.default_rng(41)
    prims, secs = [], []
    for _ in range(n):
        prims.append(_row(*FLAT20))
        s = _row(*RECT16)
        s.update(pos=tuple(rng.normal(scale=0.7, size=3)), alpha=float(rng.uniform(0, 3)), beta=float(rng.uniform(0, 6)), n_len=4)
        secs.append(s)
    P, S = abi.CoilSet.from_rows(prims), abi.CoilSet.from_rows(secs)
    what = abi.PAIR_M | abi.PAIR_FT | abi.PAIR_DM
    ref, _ = ctx.pairs(P, S, n, what, abi.FP64_IEEE)
    for flags in (0, abi.FAR_FIELD):
        got, _ = ctx.pairs(P, S, n, what, abi.FP64, flags)
        for k, v in ref.items():   # some nodes lie next to the winding: rounding of terms up to a thousand times the sum
            assert np.max(np.abs(got[k] - v)) <= 1e-10 * np.max(np.abs(v)), (k, flags)
    Mr, Gr, _ = ctx.pairs_grad(P, S, n, abi.FP64_IEEE)
    Mg, Gg, _ = ctx.pairs_grad(P, S, n, abi.FP64)
    assert np.max(np.abs(Mg - Mr)) <= 1e-10 * np.max(np.abs(Mr)) and np.max(np.abs(Gg - Gr)) <= 1e-10 * np.max(np.abs(Gr))


def test_pairs_no_slower_than_ieee(ctx):
    """2,048 pairs of a short slow rule with filaments, whose few nodes leave the set-up of a node to show."""
    rng, n = np.random.default_rng(41), 2048
    prims, secs = [], []
    for _ in range(n):
        prims.append(_row(*FLAT20))
        s = _row("FILAMENT", 0.25, 0.0, 0.0, 80, 1)
        s.update(pos=tuple(rng.normal(scale=0.2, size=3)), alpha=float(rng.uniform(0, 3)), beta=float(rng.uniform(0, 6)), n_len=1)
        secs.append(s)
    P, S = abi.CoilSet.from_rows(prims), abi.CoilSet.from_rows(secs)
    mf = abi.PAIR_M | abi.PAIR_FT
    ms = {p: min(ctx.pairs(P, S, n, mf, p)[1].kernel_ms for _ in range(9)) for p in (abi.FP64, abi.FP64_IEEE)}
    print(f"\n{n} pairs: {1e3 * ms[abi.FP64]:.0f} us, IEEE {1e3 * ms[abi.FP64_IEEE]:.0f}")
    assert ms[abi.FP64] <= ms[abi.FP64_IEEE]


def test_pairs_grad_fp32c_time(ctx):
    """32 pairs next to each other's windings: each work item ends with a few nodes for the FP64 rule, after all its nodes
    in float; half as long again as IEEE arithmetic at all of them is room for both."""
    rng, n = np.random.default_rng(3), 32
    prims, secs = [], []
    for _ in range(n):
        prims.append(_row(*RECT16))
        s = _row(*RECT16)
        s.update(pos=tuple(rng.normal(scale=0.2, size=3)), alpha=float(rng.uniform(0, 3)), beta=float(rng.uniform(0, 6)), n_len=4)
        secs.append(s)
    P, S = abi.CoilSet.from_rows(prims), abi.CoilSet.from_rows(secs)
    ms = {p: min(ctx.pairs_grad(P, S, n, p)[2].kernel_ms for _ in range(9)) for p in (abi.FP32C, abi.FP64_IEEE)}
    print(f"\n{n} pairs: FP32C {1e3 * ms[abi.FP32C]:.0f} us, IEEE {1e3 * ms[abi.FP64_IEEE]:.0f}")
    assert ms[abi.FP32C] <= 1.5 * ms[abi.FP64_IEEE]


# the most points (times coils) that a wave each could serve, and one more: short rules, whose points have few nodes
# wherever they lie, were 1.2 times slower a wave each. Five per cent for the card
@pytest.mark.parametrize("coil,copies,n", [(FLAT20, 1, 4096), (RECT16, 2, 2048), (THIN12, 1, 2048), (RECT59, 1, 4096)])
def test_time_at_the_whole_wave_limit(ctx, coil, copies, n):
    cs = abi.CoilSet.from_rows([_row(*coil)] * copies)
    pts = np.random.default_rng(2).normal(scale=0.3, size=(n + 1, 3))
    us = [1e3 * min(ctx.fields(cs, pts[:m], abi.B, abi.FP64)[1].kernel_ms for _ in range(25)) for m in (n, n + 1)]
    print(f"\n{coil} {copies} coils: {n} points {us[0]:.1f} us, {n + 1} points {us[1]:.1f}")
    assert us[0] <= 1.05 * us[1]


# few coils of two rows, whose reduced rules end in a few long waves, and one coil of the longest rules at the fewest points
# of one lane each, which the visit order gathered in a few waves: 0.69, 0.48 and 0.29 of IEEE's time that way, and 0.59,
# 0.16 and 0.12 by own nodes and in index order
@pytest.mark.parametrize("coil,copies,n,share", [(("RECTANGULAR", 0.2, 0.02, 0.3, 63, 2), 6, 16384, 0.65),
                                                 (("RECTANGULAR", 0.1, 0.1, 0.1, 100, 100), 1, 65536, 0.3),
                                                 (("FLAT", 0.1, 0.05, 0.0, 100, 100), 1, 65536, 0.2)])
def test_time_of_few_coils(ctx, coil, copies, n, share):
    rng = np.random.default_rng(3)
    rows = []
    for _ in range(copies):
        row = _row(*coil)
        row.update(pos=tuple(rng.normal(scale=0.3 if copies > 1 else 0.0, size=3)), alpha=float(rng.uniform(0, 3)))
        rows.append(row)
    cs = abi.CoilSet.from_rows(rows)
    pts = rng.normal(scale=0.4, size=(n, 3))
    ms = {p: min(ctx.fields(cs, pts, abi.B, p)[1].kernel_ms for _ in range(9)) for p in (abi.FP64, abi.FP64_IEEE)}
    print(f"\n{coil} {copies} coils {n} points: {1e3 * ms[abi.FP64]:.0f} us, IEEE {1e3 * ms[abi.FP64_IEEE]:.0f}")
    assert ms[abi.FP64] <= share * ms[abi.FP64_IEEE]
