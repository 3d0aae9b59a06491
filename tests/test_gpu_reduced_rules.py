"""The reduced rules against the coil's own rule.

CCOIL_FP64 replaces a coil's angular or thickness sum by one of fewer nodes where the rule has converged to rounding;
CCOIL_FP64_IEEE sums the coil's own rule at every pair. Points around the winding at distances from a hundredth to
thirty times its cross-section cross every class boundary, inside the bore, beyond the ends, outside and on the axis.

Tolerance, per point and relative to the coil's own field: the reduced and the own rule each err by at most 1e-15 of the
sum of the node terms' magnitudes, and both sums carry rounding of a few ulps of it. That sum exceeds the field by at
most about (1 + y)^2 (y = D / r_max: the terms cancel to the far field) times 10 for A and B and 100 for the gradient
where eta >= 0.1 (its terms grow like eta^-4): 2e-14 (1 + y)^2 and 2e-13 (1 + y)^2. Closer points keep the own angular
rule and differ from CCOIL_FP64_IEEE as before: 1e-11 for A and B, 1e-6 for the gradient. Pairs that take the far-field
series are held to its 1e-13 of the coil's field at their distance instead.
"""
import numpy as np
import pytest

import ccoil_abi as abi
import oracle as O
import workloads as W

pytestmark = pytest.mark.gpu

COILS = [("RECTANGULAR", 0.1, 0.1, 0.1, 59, 27), ("RECTANGULAR", 0.02, 0.2, 0.01, 48, 34), ("THIN", 0.3, 0.0, 0.2, 80, 1),
         ("THIN", 0.05, 0.0, 0.005, 12, 1), ("FLAT", 0.1, 0.05, 0.0, 80, 20), ("FLAT", 0.4, 0.2, 0.0, 100, 100),
         ("FILAMENT", 0.25, 0.0, 0.0, 80, 1), ("FILAMENT", 0.25, 0.0, 0.0, 6, 1), ("RECTANGULAR", 0.2, 0.02, 0.3, 21, 2),
         ("FLAT", 0.1, 0.05, 0.0, 20, 7)]


def _row(typ, R, a, b, n_ang, n_thk):
    p = dict(type=typ, R=R, a=a, b=b, N=250, I=3.0, pos=np.array([0.03, -0.02, 0.05]), alpha=0.7, beta=1.9)
    row = W.coil_row(W.make_coil(p))
    row.update(n_ang=n_ang, n_thk=n_thk, blocks=(1, 1, 1))
    return row


def _points(rng, row, n):
    """Global points around the winding, and their r, z in the coil's frame."""
    R, a, b = row["R"], row["a"], row["b"]
    size = max(a, b, 0.05 * R)
    d = size * 10.0 ** rng.uniform(-2.0, 1.5, n)
    t = rng.uniform(0.0, 2.0 * np.pi, n)
    r = np.abs(R + a * rng.uniform(0.0, 1.0, n) + d * np.cos(t))
    z = b * rng.uniform(-0.5, 0.5, n) + d * np.sin(t)
    r[: n // 20] = R * 10.0 ** rng.uniform(-9.0, -2.0, n // 20)   # the axis
    phi = rng.uniform(0.0, 2.0 * np.pi, n)
    loc = np.stack([r * np.cos(phi), r * np.sin(phi), z], axis=1)
    return np.asarray(row["pos"]) + loc @ W.rotation(row["alpha"], row["beta"]).T, r, z


def check(ctx, row, n, prec, flags, seed):
    rng = np.random.default_rng(seed)
    pts, r, z = _points(rng, row, n)
    cs = abi.CoilSet.from_rows([row])
    q = abi.A | abi.B | abi.G
    ref, _ = ctx.fields(cs, pts, q, abi.FP64_IEEE)
    got, _ = ctx.fields(cs, pts, q, prec, flags)
    R, a, hb = row["R"], row["a"], 0.5 * row["b"] if row["use_fast"] else 0.0
    zd = np.maximum(np.abs(z) - hb, 0.0)
    rho = np.clip(np.hypot(r, zd), R, R + a)
    eta = np.arccosh(1.0 + ((rho - r) ** 2 + zd * zd) / (2.0 * rho * r))
    y = np.hypot(r, z) / np.hypot(R + a, hb)
    worst = {}
    for k, near, far in (("A", 1e-11, 2e-14), ("B", 1e-11, 2e-14), ("G", 1e-6, 2e-13)):
        err = np.linalg.norm(got[k] - ref[k], axis=1)
        scale = np.linalg.norm(ref[k], axis=1)
        # near the axis A and B_rho vanish like r while their sums' terms do not: those are of the size of B R for A
        # and of B for B_rho, which the gradient divides by r (down to 1e-5 R)
        b = np.linalg.norm(ref["B"], axis=1)
        scale += b * R if k == "A" else b / np.maximum(r, 1e-5 * R) if k == "G" else 0.0
        e = err / scale
        tol = np.where(eta > 0.1, far * (1.0 + y) ** 2, near)
        if flags & abi.FAR_FIELD:
            tol = np.maximum(tol, 1e-12)
        worst[k] = float(np.max(e / tol))
        i = int(np.argmax(e / tol))
        assert e[i] <= tol[i], (row["n_ang"], row["n_thk"], k, n, e[i], tol[i], eta[i], y[i], r[i], z[i])
    return worst


@pytest.mark.parametrize("n", [16500, 131500])
@pytest.mark.parametrize("coil", COILS, ids=lambda c: f"{c[0]}-{c[4]}x{c[5]}")
def test_records_match_the_own_rule(ctx, coil, n):
    """The record pass of the series mode: lanes grouped per record (few points), and uniform waves (many)."""
    print(f"\n{coil} n={n}: worst error over tolerance {check(ctx, _row(*coil), n, abi.FP64, abi.FAR_FIELD, 5)}")


@pytest.mark.parametrize("n_coils,n", [(1, 300), (8, 300), (9, 5000), (65, 5000), (130, 300), (23, 70000), (40, 270000),
                                       (1, 8400000)])
def test_records_of_many_coils(ctx, n_coils, n):
    """Every point next to every coil, at coil counts around the rows of eight that the records are placed in, one row and
    several, and one, a few and over 2,048 tiles of the scans: the series mode against the rule, which differ by the
    order of their sums and by rounding (1e-12 of the field's largest value)."""
    rng = np.random.default_rng(17)
    rows = []
    for k in range(n_coils):
        row = _row(*COILS[k % 8])
        row.update(pos=tuple(rng.normal(scale=0.02, size=3)), alpha=float(rng.uniform(0, 3)), beta=float(rng.uniform(0, 6)))
        rows.append(row)
    cs = abi.CoilSet.from_rows(rows)
    pts = rng.normal(scale=0.12, size=(n, 3))
    ref, _ = ctx.fields(cs, pts, abi.B, abi.FP64)
    got, _ = ctx.fields(cs, pts, abi.B, abi.FP64, abi.FAR_FIELD)
    assert np.max(np.abs(got["B"] - ref["B"])) <= 1e-12 * np.max(np.abs(ref["B"]))


LONG = [("RECTANGULAR", 0.02, 0.01, 0.6, 80, 20), ("THIN", 0.02, 0.0, 1.0, 100, 1), ("FLAT", 0.01, 0.3, 0.0, 100, 100),
        ("RECTANGULAR", 0.1, 0.05, 1e-4, 80, 2), ("RECTANGULAR", 0.3, 0.3, 0.3, 100, 100)]


@pytest.mark.parametrize("coil", LONG, ids=lambda c: f"{c[0]}-{c[2]}x{c[3]}")
def test_series_matches_the_own_rule(ctx, coil):
    """The series' moments of sheets from none to 99 % of r_max in half-length, 1 to 100 sheets, few orders to all: on
    shells of 1.3 to 40 r_max, relative to the field's largest value on the shell, the series' 1e-13 with the own rule's
    rounding of terms that cancel with the distance in radii."""
    row = _row(*coil)
    rng = np.random.default_rng(13)
    y = np.repeat(np.array([1.3, 1.6, 2.0, 3.0, 5.0, 12.0, 40.0]), 300)
    d = rng.normal(size=(y.size, 3))
    rmax = np.hypot(row["R"] + row["a"], 0.5 * row["b"])
    D = y * rmax
    pts = np.asarray(row["pos"]) + d / np.linalg.norm(d, axis=1)[:, None] * D[:, None]
    cs = abi.CoilSet.from_rows([row])
    ref, _ = ctx.fields(cs, pts, abi.A | abi.B | abi.G, abi.FP64_IEEE)
    got, _ = ctx.fields(cs, pts, abi.A | abi.B | abi.G, abi.FP64, abi.FAR_FIELD)
    for k, ulps in (("A", 2e-14), ("B", 2e-14), ("G", 2e-13)):
        err, ref_k = np.linalg.norm(got[k] - ref[k], axis=1), np.linalg.norm(ref[k], axis=1)
        for v in np.unique(y):
            s = y == v
            tol = 1e-13 + ulps * (1.0 + v * rmax / (row["R"] + row["a"])) ** 2
            assert np.max(err[s]) <= tol * np.max(ref_k[s]), (k, v, np.max(err[s]) / np.max(ref_k[s]), tol)


@pytest.mark.parametrize("n,split", [(300, 16), (600, 64), (5000, 16), (20000, 4), (70000, 1)])
@pytest.mark.parametrize("coil", COILS, ids=lambda c: f"{c[0]}-{c[4]}x{c[5]}")
def test_field_kernel_matches_the_own_rule(ctx, coil, n, split):
    """The rule alone at every launch shape: a whole wave, 16 or 4 lanes per point, one lane per point."""
    row = _row(*coil)
    _, rep = ctx.fields(abi.CoilSet.from_rows([row]), np.zeros((n, 3)), abi.B, abi.FP64)
    assert rep.split == split
    print(f"\n{coil} n={n}: worst error over tolerance {check(ctx, row, n, abi.FP64, 0, 7)}")


@pytest.mark.parametrize("blocks", [(1, 1, 1), (3, 2, 2)])
@pytest.mark.parametrize("coil", COILS, ids=lambda c: f"{c[0]}-{c[4]}x{c[5]}")
def test_pairs_match_the_own_rule(ctx, coil, blocks):
    """M, F, T, dM and the gradient of M of one primary with secondaries from inside its bore and across its winding to
    twenty radii away, CCOIL_FP64 against CCOIL_FP64_IEEE, alone (a few work items) and as a batch. Each sum's terms
    exceed it by at most about a thousand here (M relative to its size over the pose's neighbourhood), and both rules
    round each term to a few ulps: 1e-12, and 1e-10 where the secondary crosses the primary's winding. The derivatives
    with respect to the primary's geometry cancel once more like the field they come from, by (1 + y)^2 / 10 beyond."""
    row = _row(*coil)
    rng = np.random.default_rng(11)
    size = np.hypot(row["R"] + row["a"], 0.5 * row["b"])
    secs = []
    ys = np.array([0.3, 0.9, 1.6, 2.5, 4.0, 8.0, 20.0])
    for y in ys:
        d = rng.standard_normal(3)
        s = _row("RECTANGULAR", 0.3 * row["R"], 0.1 * row["R"], 0.2 * row["R"], 14, 3)
        s.update(pos=tuple(np.asarray(row["pos"]) + y * size * d / np.linalg.norm(d)), alpha=rng.uniform(0, 3.0),
                 beta=rng.uniform(0, 6.0), n_len=5, blocks=blocks)
        secs.append(s)
    P, S, n = abi.CoilSet.from_rows([row]), abi.CoilSet.from_rows(secs), len(secs)
    what, prim = abi.PAIR_M | abi.PAIR_FT | abi.PAIR_DM, np.zeros(n, dtype=np.int64)
    ref, _ = ctx.pairs(P, S, n, what, abi.FP64_IEEE, prim_index=prim)
    got, _ = ctx.pairs(P, S, n, what, abi.FP64, prim_index=prim)
    Mr, Gr, _ = ctx.pairs_grad(P, S, n, abi.FP64_IEEE, prim_index=prim)
    Mg, Gg, _ = ctx.pairs_grad(P, S, n, abi.FP64, prim_index=prim)
    one, _ = ctx.pairs(P, S, 1, what, abi.FP64, prim_index=prim[:1], sec_index=np.array([3]))
    norm = np.linalg.norm
    dist = np.array([norm(np.array(s["pos"]) - np.array(row["pos"])) for s in secs])
    mscale = np.abs(ref["M"]) + norm(ref["dM"], axis=1) * dist
    errs = {"M": np.abs(got["M"] - ref["M"]) / mscale, "M of grad": np.abs(Mg - Mr) / mscale,
            "grad": norm(Gg - Gr, axis=1) / norm(Gr, axis=1)}
    for k in ("F", "T", "dM"):
        errs[k] = norm(got[k] - ref[k], axis=1) / norm(ref[k], axis=1)
    print(f"\n{coil} {blocks}: " + ", ".join(f"{k} {v.max():.2g}" for k, v in errs.items()))
    for k, v in errs.items():
        tol = np.where(ys < 1.0, 1e-10, 1e-12 * (np.maximum(1.0, (1.0 + ys) ** 2 / 10.0) if k == "grad" else 1.0))
        assert np.all(v <= tol), (k, v, tol)
    assert abs(one["M"][0] - ref["M"][3]) <= 1e-12 * mscale[3]
    assert norm(one["F"][0] - ref["F"][3]) <= 1e-12 * norm(ref["F"][3])


@pytest.mark.parametrize("n", [63, 5000])
@pytest.mark.parametrize("coil", COILS, ids=lambda c: f"{c[0]}-{c[4]}x{c[5]}")
def test_adjoint_matches_the_own_rule(ctx, coil, n):
    """The nine derivatives of an objective of B at points of every class but the own angular rule's, waves of mixed
    classes among them. Each point's terms agree to 2e-13 (1 + y)^2 of its gradient (above); the points' sum cancels by
    at most the square root of their number here: 1e-10."""
    row = _row(*coil)
    rng = np.random.default_rng(13)
    pts, r, z = _points(rng, row, 4 * n)
    R, a, hb = row["R"], row["a"], 0.5 * row["b"] if row["use_fast"] else 0.0
    zd = np.maximum(np.abs(z) - hb, 0.0)
    rho = np.clip(np.hypot(r, zd), R, R + a)
    keep = (((rho - r) ** 2 + zd * zd > 0.01 * rho * r) & (r > 0.01 * R) & (np.hypot(r, z) < 10 * np.hypot(R + a, hb)))
    pts = np.ascontiguousarray(pts[keep][:n])
    g = rng.standard_normal(pts.shape)
    cs = abi.CoilSet.from_rows([row])
    ref, _ = ctx.field_gradient(cs, pts, g, abi.FP64_IEEE)
    got, _ = ctx.field_gradient(cs, pts, g, abi.FP64)
    err = np.abs(got - ref) / np.maximum(np.abs(ref), 1e-3 * np.max(np.abs(ref) * [row["current"], R, a, row["b"], R, R, R, 1, 1]) /
                                         np.array([row["current"], R, max(a, 1e-3 * R), max(row["b"], 1e-3 * R), R, R, R, 1, 1]))
    print(f"\n{coil} {len(pts)} points: {err.max():.2g}")
    assert err.max() <= 1e-10


COAXIAL = [(0.1, 0.05, 0.12, 0.1, 0.03, 0.05), (0.05, 0.0, 0.2, 0.07, 0.04, 0.01), (0.2, 0.1, 0.02, 0.02, 0.0, 0.3),
           (0.1, 0.01, 0.1, 0.12, 0.02, 0.1), (0.03, 0.02, 0.1, 0.2, 0.1, 0.1)]   # R, a, b of both


@pytest.mark.parametrize("apart", [0, 1])
@pytest.mark.parametrize("i", range(len(COAXIAL)))
def test_coaxial_pairs(ctx, i, apart):
    """M and axial force against the long double sum of the coils' own rules, single and of several blocks, at axial gaps
    of a hundredth to thirty radii, and side by side (nested) at small offsets. The angular sum cancels to at most some
    1/100 of its terms, the offsets keep the force off its zero at the middle: 1e-12 of the value. The oracle's long double
    sum itself cancels from eight terms of up to z log(2 z / D) (force: of four logarithms), weights 2 t r: some 2^-60 of
    20 |z| (20) times them."""
    R, a, b, R2, a2, b2 = COAXIAL[i]
    rows, orders, coils = ([], []), [], ([], [])
    gaps = np.geomspace(0.01, 30.0, 24) * max(R, R2) + 0.5 * (b + b2) if apart else np.linspace(0.3, 0.9, 8) * max(b, b2)
    for n, d in enumerate(gaps):
        p = O.make_coil(R, a, b, 250, 3.0, pos=(0, 0, 0.1))
        s = O.make_coil(R2, a2, b2, 100, -2.0, pos=(0, 0, 0.1 + (d if n % 2 else -d)))
        blocks = 1 + n % 3 // 2
        args = np.array([blocks, blocks if a else 1, 1, 80, 20 if a else 1, 20] + [1, blocks if a2 else 1, 1, 80, 20 if a2 else 1, 20])
        orders.append(args)
        for c, part, half in ((p, 0, args[:6]), (s, 1, args[6:])):
            coils[part].append(c)
            rows[part].append(dict(use_fast=int(c.use_fast), n_ang=int(half[3]), n_thk=int(half[4]), n_len=int(half[5]),
                                   blocks=tuple(int(v) for v in half[:3]), R=c.R, a=c.a, b=c.b, J=c.J, current=c.I,
                                   turns=float(c.N), frequency=c.freq, pos=tuple(c.pos), alpha=0.0, beta=0.0))
    P, S = (abi.CoilSet.from_rows(r) for r in rows)
    out, _ = ctx.pairs_zaxis(P, S, len(orders), abi.PAIR_M | abi.PAIR_FT)
    for k, (p, s, args) in enumerate(zip(*coils, orders)):
        m, f = O.mutual_inductance_zaxis_fast(p, s, args, True), O.force_zaxis_fast(p, s, args, True)
        lost = 2.0 ** -60 * 20.0 * 2e-7 * np.pi ** 2 * abs(p.J * s.J) * p.a * s.a * (p.R + p.a) * (s.R + s.a)
        assert abs(out["M"][k] - m) <= 1e-12 * abs(m) + lost * gaps[k] / abs(p.I * s.I), (k, gaps[k])
        assert abs(out["Fz"][k] - f) <= 1e-12 * abs(f) + lost, (k, gaps[k])


@pytest.mark.parametrize("R,a,b", [(1e21, 1e21, 1e21), (1e-22, 1e-22, 1e-22), (1e-3, 0.0, 1e5), (1.0, 1e-7, 0.5), (2.0, 1e-3, 1e5)])
def test_classes_out_of_floats_range(ctx, R, a, b):
    """Coils whose points' classes float cannot tell: too large or small to square, far longer than wide, far thinner. At
    points in and around the winding, and at its end, CCOIL_FP64 and CCOIL_FP64_IEEE differ by the rounding of their node
    terms: 1e-11 of the largest value."""
    row = _row("RECTANGULAR" if a else "THIN", R, a, b, 80, 20 if a else 1)
    row.update(pos=(0.0, 0.0, 0.0), alpha=0.0, beta=0.0)
    rng = np.random.default_rng(19)
    n, phi = 1000, rng.uniform(0, 2 * np.pi, 1000)
    r = np.where(np.arange(n) % 2, R + max(a, 1e-3 * R) * rng.uniform(-1, 2, n), R * rng.uniform(0.5, 3, n))
    z = np.where(np.arange(n) % 3, b * rng.uniform(-0.5, 0.5, n), 0.5 * b + R * rng.uniform(-1, 1, n))
    pts = np.stack([r * np.cos(phi), r * np.sin(phi), z], axis=1)
    cs = abi.CoilSet.from_rows([row])
    ref, _ = ctx.fields(cs, pts, abi.A | abi.B, abi.FP64_IEEE)
    got, _ = ctx.fields(cs, pts, abi.A | abi.B, abi.FP64)
    for k in ("A", "B"):
        assert np.all(np.isfinite(ref[k]))
        assert np.max(np.abs(got[k] - ref[k])) <= 1e-11 * np.max(np.abs(ref[k])), k


@pytest.mark.parametrize("a,b", [(1e-3, 1e4), (1e-2, 200.0)])
def test_end_of_a_long_thin_coil(ctx, a, b):
    """Where float coordinates are as coarse as the winding is thick: points within two thicknesses of its end. The FP64
    rules agree there to the rounding of their node terms, as above: 1e-11 of the largest value."""
    row = _row("RECTANGULAR", 1.0, a, b, 80, 30)
    row.update(pos=(0.0, 0.0, 0.0), alpha=0.0, beta=0.0)
    rng = np.random.default_rng(29)
    n = 1000
    phi, r, z = rng.uniform(0, 2 * np.pi, n), 1.0 + a * rng.uniform(-1, 2, n), 0.5 * b + a * rng.uniform(-2, 2, n)
    pts = np.stack([r * np.cos(phi), r * np.sin(phi), z], axis=1)
    cs = abi.CoilSet.from_rows([row])
    ref, _ = ctx.fields(cs, pts, abi.A | abi.B, abi.FP64_IEEE)
    got, _ = ctx.fields(cs, pts, abi.A | abi.B, abi.FP64)
    for k in ("A", "B"):
        assert np.max(np.abs(got[k] - ref[k])) <= 1e-11 * np.max(np.abs(ref[k])), k
