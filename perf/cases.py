"""Performance cases: the calls a program makes through this framework's public entry points, with the sizes its tests,
its benchmark and its planner use.

  field      Context.fields on device pointers: A, B, E or the gradient of one coil or a coil group over points
  dropin     the c_coil module on numpy arrays, as a program written for the reference calls it (FP32C, its default)
  design     a coil-design step: B through ccoil_torch's autograd function and the gradient of an objective of it
  pairs      Context.pairs: M, force and torque, and dM/dp of many coil pairs (own coils per pair, uneven orders), or
             of the off-diagonal entries of a coil matrix
  pairs_grad Context.pairs_grad: M and its 16 parameter derivatives
  coaxial    Context.pairs_zaxis: M and axial force of coaxial pairs

Modes: fp64 (the rule in double), fp64_far (CCOIL_FAR_FIELD: the series beyond each coil's far-field distance), fp32c.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "c-coil_amd"))

import ccoil_abi as abi  # noqa: E402
import ccoil_torch  # noqa: E402
import workloads as W  # noqa: E402

BITS = {"A": abi.A, "B": abi.B, "E": abi.E, "G": abi.G}
WIDTH = {"A": 3, "B": 3, "E": 3, "G": 9}
MODES = {"fp64": (abi.FP64, 0), "fp64_far": (abi.FP64, abi.FAR_FIELD), "fp32c": (abi.FP32C, 0)}
WHAT = {"M": abi.PAIR_M, "F": abi.PAIR_FT, "D": abi.PAIR_DM}
MAX_EXACT_NODES = 1.2e10   # node evaluations that exact() does in a few seconds


def listed():
    return [
        # one coil in a control loop or a sensor model: the call's latency
        dict(name="field_1x4096_b", kind="field", coils=1, points=4096, q="B", mode="fp64"),
        # a small assembly probed at a few odd places, every quantity
        dict(name="field_5x777_abeg", kind="field", coils=5, points=777, q="ABEG", mode="fp64"),
        # a reference map by the rule alone (the library's accurate default)
        dict(name="field_64x131072_bg", kind="field", coils=64, points=131072, q="BG", mode="fp64"),
        # a ragged map just above the size where points are sorted
        dict(name="field_128x16411_bg_far", kind="field", coils=128, points=16411, q="BG", mode="fp64_far"),
        # the benchmark's workload
        dict(name="field_128x1M_bg_far", kind="field", coils=128, points=1 << 20, q="BG", mode="fp64_far"),
        # the fast mode, which is the C ABI front end's and the module's default
        dict(name="field_128x262145_bg_fp32c", kind="field", coils=128, points=262145, q="BG", mode="fp32c"),
        # the reference's Python API on host arrays
        dict(name="dropin_12x20011_a", kind="dropin", coils=12, points=20011, q="A"),
        # one step of a gradient-based coil design
        dict(name="design_64x4096", kind="design", coils=64, points=4096),
        # one pair, as a program that places two coils asks for it
        dict(name="pairs_1_mf", kind="pairs", pairs=1, what="MF", mode="fp64"),
        # a batch of uneven pairs with the series
        dict(name="pairs_8192_mf_far", kind="pairs", pairs=8192, what="MF", mode="fp64_far"),
        # sensitivity of couplings to every parameter
        dict(name="pairs_grad_256", kind="pairs_grad", pairs=256),
        # a table of coaxial assemblies
        dict(name="coaxial_1500", kind="coaxial", pairs=1500),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["field"] * 5 + ["dropin", "design", "pairs", "pairs", "matrix", "pairs_grad", "coaxial"])
    if kind == "field":
        mode = rng.choice(["fp64", "fp64_far", "fp32c"])
        coils = _log(rng, 1, 128)
        # coil-points of the rule alone up to the listed map's, of the series modes up to the benchmark's
        most = min(1 << 20, (1 << 23 if mode == "fp64" else 1 << 27) // coils)
        return dict(kind="field", coils=coils, points=_log(rng, 256, most), q=rng.choice(["B", "BG", "A", "AE", "G", "ABEG"]),
                    mode=mode)
    if kind == "dropin":
        return dict(kind="dropin", coils=_log(rng, 1, 24), points=_log(rng, 500, 40000), q=rng.choice(["B", "A", "G"]))
    if kind == "design":
        return dict(kind="design", coils=_log(rng, 4, 96), points=_log(rng, 256, 8192))
    if kind == "pairs":
        return dict(kind="pairs", pairs=_log(rng, 1, 4096), what=rng.choice(["M", "MF", "F", "MFD"]),
                    mode=rng.choice(["fp64", "fp64_far", "fp32c"]))
    if kind == "matrix":
        return dict(kind="pairs", matrix=_log(rng, 4, 48), what=rng.choice(["M", "MFD"]),
                    mode=rng.choice(["fp64", "fp64_far"]))
    if kind == "pairs_grad":
        return dict(kind="pairs_grad", pairs=_log(rng, 1, 256))
    return dict(kind="coaxial", pairs=_log(rng, 1, 4096))


# ---- inputs --------------------------------------------------------------------------------------------------------

_context = None


def _ctx():
    """The program's library context, on torch's stream; a program keeps one."""
    global _context
    if _context is None:
        _context = abi.Context(0)
        _context.set_stream(torch.cuda.current_stream().cuda_stream)
    return _context


def _coils(case, seed):
    """(coil parameters, their rows with planned orders, points) of a field, drop-in or design case."""
    n = case["points"]
    if case["kind"] == "design":
        params, pts = W.adjoint_workload(case["coils"], n, seed=seed)
        for p in params:
            p["R"] += 0.08   # bores that clear the target region, whatever their offset and tilt
    elif case["coils"] == 1:
        params, pts = W.single_rect_workload(n, seed=seed)
        params[0]["I"] = 1.0 + 0.01 * (seed % 100)
    else:
        params, pts = W.group_workload(case["coils"], n, seed=seed)
    return params, W.group_rows(params), pts


def _pair_rows(case, seed):
    """(primary rows, secondary rows, primary index, secondary index) of a pair case."""
    if case["kind"] == "coaxial":
        _, _, prim, sec = W.coaxial_workload(case["pairs"], seed=seed)
        return prim, sec, None, None
    if "matrix" in case:
        params = W.random_coil_params(np.random.default_rng(seed), case["matrix"])
        i, j = W.matrix_pairs(case["matrix"])
        return W.group_rows(params), W.secondary_rows(params), i, j
    prim, sec = W.pair_workload(case["pairs"], seed=seed)
    return prim, sec, None, None


def prepare(case, seed):
    ctx = _ctx()
    s = dict(case=case, ctx=ctx)
    kind = case["kind"]
    if kind in ("field", "dropin", "design"):
        params, rows, pts = _coils(case, seed)
        if kind == "dropin":
            import c_coil
            C = c_coil.coil
            coils = [W.make_coil(p) for p in params]
            s.update(C=C, pts=pts, group=c_coil.coil_group.CoilGroup(coils, C.PrecisionFactor(5.0)))
            return s
        s["pts"] = torch.from_numpy(pts).cuda()
        if kind == "design":
            s["model"] = ccoil_torch.CoilFieldModel(rows, ctx, abi.FP64)
            s["params"] = s["model"].initial_params().requires_grad_(True)
            g = np.random.default_rng(seed + 1).standard_normal(pts.shape) / len(pts)   # dL/dB of the objective
            s["g"] = torch.from_numpy(g).cuda()
            return s
        s["coils"] = abi.CoilSet.from_rows(rows)
        s["q"] = sum(BITS[k] for k in case["q"])
        s["out"] = {k: torch.empty((len(pts), WIDTH[k]), dtype=torch.float64, device="cuda") for k in case["q"]}
        return s
    prim, sec, i, j = _pair_rows(case, seed)
    s.update(P=abi.CoilSet.from_rows(prim), S=abi.CoilSet.from_rows(sec), i=i, j=j, n=len(prim) if i is None else len(i))
    if kind == "pairs":
        s["what"] = sum(WHAT[k] for k in case["what"])
        wide = dict(M=("M",), F=("F", "T"), D=("dM",))
        s["out"] = {k: torch.empty((s["n"],) if k == "M" else (s["n"], 3), dtype=torch.float64, device="cuda")
                    for w in case["what"] for k in wide[w]}
    elif kind == "coaxial":
        s["out"] = {k: torch.empty(s["n"], dtype=torch.float64, device="cuda") for k in ("M", "Fz")}
    return s


def run(s):
    case, ctx, kind = s["case"], s["ctx"], s["case"]["kind"]
    if kind == "field":
        prec, flags = MODES[case["mode"]]
        return ctx.fields(s["coils"], s["pts"], s["q"], prec, flags | abi.DEVICE_POINTERS, out=s["out"])[0]
    if kind == "dropin":
        f = {"A": s["group"].compute_all_A_potential_vectors, "B": s["group"].compute_all_B_field_vectors,
             "G": s["group"].compute_all_B_gradient_matrices}[case["q"]]
        return f(s["pts"], s["C"].GPU)
    if kind == "design":
        B = s["model"].B(s["params"], s["pts"])
        (grad,) = torch.autograd.grad(B, s["params"], s["g"])
        return {"B": B, "grad": grad}
    if kind == "pairs":
        prec, flags = MODES[case["mode"]]
        return ctx.pairs(s["P"], s["S"], s["n"], s["what"], prec, flags | abi.DEVICE_POINTERS, prim_index=s["i"],
                         sec_index=s["j"], out=s["out"])[0]
    if kind == "pairs_grad":
        M, grad, _ = ctx.pairs_grad(s["P"], s["S"], s["n"], abi.FP64)
        return {"M": M, "grad": grad}
    return ctx.pairs_zaxis(s["P"], s["S"], s["n"], abi.PAIR_M | abi.PAIR_FT, abi.DEVICE_POINTERS, out=s["out"])[0]


def work(case):
    """Inputs and outputs once each; per (coil, point), or per pair and secondary ring direction, the least that an
    evaluation by any expansion takes: the change of frame there and back and some eight terms of each sum."""
    kind = case["kind"]
    if kind in ("field", "dropin", "design"):
        width = sum(WIDTH[k] for k in case.get("q", "B"))
        flops = 60 + 8 * 4 * width + 9 * width
        n, c = case["points"], case["coils"]
        grad = 9 * c if kind == "design" else 0
        passes = 3 if kind == "design" else 1   # forward, and B and its gradient again for the adjoint
        return {"bytes": 8.0 * (n * (3 + width + (6 if kind == "design" else 0)) + 40 * c + grad),
                "flops": float(flops) * n * c * passes}
    n = case["pairs"] if "pairs" in case else case["matrix"] * (case["matrix"] - 1)
    if kind == "coaxial":
        return {"bytes": 8.0 * n * (40 + 2), "flops": 8.0 ** 3 * 60 * n}   # eight nodes in each of three dimensions
    out = 17 if kind == "pairs_grad" else sum({"M": 1, "F": 6, "D": 3}[k] for k in case["what"])
    return {"bytes": 8.0 * n * (40 + out), "flops": 8.0 ** 2 * (60 + 32 * out) * n}   # eight nodes around, eight across


# ---- the same rules in plain torch, 64 bits --------------------------------------------------------------------------

_dev = "cuda" if torch.cuda.is_available() else "cpu"
_rules = {}


def _gl(n):
    if n not in _rules:
        x, w = np.polynomial.legendre.leggauss(n)
        _rules[n] = torch.tensor(x, device=_dev), torch.tensor(w, device=_dev)
    return _rules[n]


def _frame(al, be):
    """Columns of the coil's frame: Rz(beta) Ry(alpha) Rz(beta)."""
    ca, sa, cb, sb = torch.cos(al), torch.sin(al), torch.cos(be), torch.sin(be)
    return torch.stack([torch.stack([cb * cb * ca - sb * sb, -sb * cb * ca - sb * cb, cb * sa]),
                        torch.stack([sb * cb * ca + sb * cb, cb * cb - sb * sb * ca, sb * sa]),
                        torch.stack([-sa * cb, sa * sb, ca])])


def _local(row, par, x, want):
    """Sums of the coil's rule at global points x (n, 3): dict of A, Bh, Bz, RP, RR, RZ, ZZ as wanted, and r, cos, sin
    of the azimuth. par: (I, R, a, b, x, y, z, alpha, beta) as tensors."""
    I, R, a, b = par[:4]
    T = _frame(par[7], par[8])
    loc = (x - par[4:7]) @ T
    z, r = loc[:, 2], torch.sqrt(loc[:, 0] ** 2 + loc[:, 1] ** 2)
    xt, wt = _gl(row["n_thk"])
    xa, wa = _gl(row["n_ang"])
    phi = 0.5 * math.pi * (1 + xa)
    c = torch.cos(phi)[None, None, :]
    one_c = 2 * torch.sin(0.5 * phi)[None, None, :] ** 2
    rho = (R + 0.5 * a * (1 + xt))[None, :, None]
    rr, zz = r[:, None, None], z[:, None, None]
    NI = row["turns"] * I * (1e-7 * 0.5 * math.pi)
    w = wt[None, :, None] * wa[None, None, :] * rho
    M = (rho - rr) ** 2 + 2 * rho * rr * one_c
    o = dict(T=T, r=r, cph=loc[:, 0] / r, sph=loc[:, 1] / r)
    if row["use_fast"]:
        w = w * (NI / b)
        z1, z2 = zz + 0.5 * b, zz - 0.5 * b
        if "A" in want:
            q = torch.sqrt(M)
            o["A"] = (w * c * (torch.asinh(z1 / q) - torch.asinh(z2 / q))).sum((1, 2))
        if "B" in want or "G" in want:
            K1, K2 = (M + z1 * z1).rsqrt(), (M + z2 * z2).rsqrt()
            dK = -2 * b * zz * (K1 * K2) ** 2 / (K1 + K2)            # K1 - K2
            h = z1 * K1 - z2 * K2
            o["Bh"] = -(w * c * dK).sum((1, 2))
            o["Bz"] = (w * (rho - rr * c) / M * h).sum((1, 2))
        if "G" in want:
            dL = dK * (K1 * K1 + K1 * K2 + K2 * K2)                  # K1^3 - K2^3
            h3 = z1 * K1 ** 3 - z2 * K2 ** 3
            o["RR"] = (w * c * (rr - rho * c) * dL).sum((1, 2))
            o["ZZ"] = (w * (rho - rr * c) * dL).sum((1, 2))
            N = -(rho - rr * c) * (rr - rho * c)
            o["RZ"] = (w * ((-c / M + 2 * N / M ** 2) * h + N / M * h3)).sum((1, 2))
    else:
        w = w * NI
        J = M + zz * zz
        K = J.rsqrt()
        if "A" in want:
            o["A"] = (w * c * K).sum((1, 2))
        if "B" in want or "G" in want:
            K3 = K ** 3
            o["Bh"] = z * (w * c * K3).sum((1, 2))
            o["Bz"] = (w * (rho - rr * c) * K3).sum((1, 2))
        if "G" in want:
            K5 = K ** 5
            o["RR"] = -3 * z * (w * c * (rr - rho * c) * K5).sum((1, 2))
            o["ZZ"] = -3 * z * (w * (rho - rr * c) * K5).sum((1, 2))
            o["RZ"] = (w * (-c * J - 3 * (rho - rr * c) * (rr - rho * c)) * K5).sum((1, 2))
    if "G" in want:
        o["RP"] = o["Bh"] / r
    return o


def _par(row, grad=False):
    p = torch.tensor([row["current"], row["R"], row["a"], row["b"], *row["pos"], row["alpha"], row["beta"]],
                     dtype=torch.float64, device=_dev)
    return p.requires_grad_(grad)


def _vec(o, u, v, k):
    """Local (radial u, azimuthal v, axial k) vectors in the global frame."""
    return torch.stack([u * o["cph"] - v * o["sph"], u * o["sph"] + v * o["cph"], k], 1) @ o["T"].T


def _exact_fields(rows, pts, q):
    x = torch.tensor(pts, device=_dev)
    out = {k: torch.zeros((len(pts), WIDTH[k]), dtype=torch.float64, device=_dev) for k in q}
    want = set(q) | ({"A"} if "E" in q else set())
    for row in rows:
        par = _par(row)
        step = max(1, (1 << 24) // (row["n_thk"] * row["n_ang"]))
        for i in range(0, len(pts), step):
            o = _local(row, par, x[i:i + step], want)
            zero = torch.zeros_like(o["r"])
            if "A" in want:
                A = _vec(o, zero, o["A"], zero)
                if "A" in q:
                    out["A"][i:i + step] += A
                if "E" in q:
                    out["E"][i:i + step] += 2 * math.pi * row["frequency"] * A
            if "B" in q:
                out["B"][i:i + step] += _vec(o, o["Bh"], zero, o["Bz"])
            if "G" in q:
                c, s = o["cph"], o["sph"]
                xy = c * s * (o["RR"] - o["RP"])
                g = torch.stack([o["RR"] * c * c + o["RP"] * s * s, xy, o["RZ"] * c,
                                 xy, o["RR"] * s * s + o["RP"] * c * c, o["RZ"] * s,
                                 o["RZ"] * c, o["RZ"] * s, o["ZZ"]], 1).reshape(-1, 3, 3)
                out["G"][i:i + step] += (o["T"] @ g).reshape(-1, 9)
    return out


def _exact_design(rows, pts, g):
    x, g = torch.tensor(pts, device=_dev), torch.tensor(g, device=_dev)
    B = torch.zeros_like(x)
    grads = []
    for row in rows:
        par = _par(row, grad=True)
        grad = torch.zeros(9, dtype=torch.float64, device=_dev)
        step = max(1, (1 << 22) // (row["n_thk"] * row["n_ang"]))
        for i in range(0, len(pts), step):
            o = _local(row, par, x[i:i + step], {"B"})
            b = _vec(o, o["Bh"], torch.zeros_like(o["r"]), o["Bz"])
            grad += torch.autograd.grad((b * g[i:i + step]).sum(), par)[0]
            B[i:i + step] += b.detach()
        grads.append(grad)
    return {"B": B, "grad": torch.stack(grads)}


def _sec_nodes(p, s, sp):
    """The secondary's nodes in chunks: weight, arm from its centre, unit tangent; sp: the secondary's parameters."""
    (xa, wa), (xt, wt), (xl, wl) = _gl(s["n_ang"]), _gl(s["n_thk"]), _gl(s["n_len"])
    phi = (math.pi * (1 + xa))[None, None, :]
    grid = torch.broadcast_tensors(phi, xt[None, :, None], xl[:, None, None],
                                   0.125 * wl[:, None, None] * wt[None, :, None] * wa[None, None, :])
    phi, gt, gl, w = (t.reshape(-1) for t in grid)
    step = max(64, (1 << 23) // (p["n_thk"] * p["n_ang"]))
    for i in range(0, len(phi), step):
        f, t, l, wi = (v[i:i + step] for v in (phi, gt, gl, w))
        ca, sa, cb, sb = torch.cos(sp[7]), torch.sin(sp[7]), torch.cos(sp[8]), torch.sin(sp[8])
        u = torch.stack([cb * ca, sb * ca, -sa])
        v = torch.stack([-sb, cb, torch.zeros_like(sb)])
        ax = torch.stack([sa * cb, sa * sb, ca])
        rho, ell = sp[1] + 0.5 * sp[2] * (1 + t), 0.5 * sp[3] * l
        c, q = torch.cos(f)[:, None], torch.sin(f)[:, None]
        yield wi * rho, ell[:, None] * ax + rho[:, None] * (c * u + q * v), c * v - q * u


def _exact_pairs(prim, sec, i, j):
    n = len(prim) if i is None else len(i)
    out = {k: torch.zeros((n,) if k == "M" else (n, 3), dtype=torch.float64, device=_dev) for k in ("M", "F", "T")}
    for k in range(n):
        p, s = (prim[k], sec[k]) if i is None else (prim[i[k]], sec[j[k]])
        pp, sp = _par(p), _par(s)
        for w, arm, tan in _sec_nodes(p, s, sp):
            o = _local(p, pp, sp[4:7] + arm, {"A", "B"})
            zero = torch.zeros_like(o["r"])
            out["M"][k] += (w * (_vec(o, zero, o["A"], zero) * tan).sum(1)).sum()
            f = w[:, None] * torch.linalg.cross(tan, _vec(o, o["Bh"], zero, o["Bz"]))
            out["F"][k] += f.sum(0)
            out["T"][k] += torch.linalg.cross(arm, f).sum(0)
        out["M"][k] *= 2 * math.pi * s["turns"] / p["current"]
        out["F"][k] *= 2 * math.pi * s["turns"] * s["current"]
        out["T"][k] *= 2 * math.pi * s["turns"] * s["current"]
    return out


def _exact_pairs_grad(prim, sec):
    M = torch.zeros(len(prim), dtype=torch.float64, device=_dev)
    G = torch.zeros((len(prim), 16), dtype=torch.float64, device=_dev)
    for k, (p, s) in enumerate(zip(prim, sec)):
        pp, sp = _par(p, grad=True), _par(s, grad=True)
        for w, arm, tan in _sec_nodes(p, s, sp):
            o = _local(p, pp, sp[4:7] + arm, {"A"})
            zero = torch.zeros_like(o["r"])
            m = (w * (_vec(o, zero, o["A"], zero) * tan).sum(1)).sum() * (2 * math.pi * s["turns"] / p["current"])
            gp, gs = torch.autograd.grad(m, (pp, sp))
            M[k] += m.detach()
            for at, d in ((0, gs), (8, gp)):
                G[k, at:at + 8] += d[torch.tensor([4, 5, 6, 7, 8, 1, 2, 3], device=_dev)]
    return {"M": M, "grad": G}


def _exact_coaxial(prim, sec):
    M = torch.zeros(len(prim), dtype=torch.float64, device=_dev)
    F = torch.zeros_like(M)

    def composite(blocks, n, lo, width):
        x, w = _gl(n)
        h = width / blocks
        mid = lo + h * (torch.arange(blocks, device=_dev, dtype=torch.float64) + 0.5)
        return (mid[:, None] + 0.5 * h * x[None, :]).reshape(-1), (0.5 * h * w).repeat(blocks)

    for k, (p, s) in enumerate(zip(prim, sec)):
        f, wf = composite(p["blocks"][0], p["n_ang"], 0.0, math.pi)
        t, wt = composite(p["blocks"][1], p["n_thk"], p["R"], p["a"])
        r, wr = composite(s["blocks"][1], s["n_thk"], s["R"], s["a"])
        t, r, c, sc = t[:, None, None], r[None, :, None], torch.cos(f), 2 * torch.sin(0.5 * f) ** 2
        w = wt[:, None, None] * wr[None, :, None] * wf * 2 * t * r * c
        D2 = (t - r) ** 2 + 2 * t * r * sc
        D = torch.sqrt(D2)
        d, hs, hp = s["pos"][2] - p["pos"][2], 0.5 * s["b"], 0.5 * p["b"]
        zs = (d + hs + hp, d + hs - hp, d - hs - hp, d - hs + hp)
        as_ = [torch.asinh(z / D) for z in zs]
        h = [z * v - torch.sqrt(D2 + z * z) for z, v in zip(zs, as_)]
        J = 1e-7 * p["J"] * s["J"]
        M[k] = (w * ((h[0] - h[1]) + (h[2] - h[3]))).sum() * (2 * math.pi * J / (p["current"] * s["current"]))
        F[k] = (w * ((as_[1] - as_[0]) + (as_[3] - as_[2]))).sum() * (-2 * math.pi * J)
    return {"M": M, "Fz": F}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("field", "dropin", "design"):
        _, rows, pts = _coils(case, seed)
        if sum(r["n_ang"] * r["n_thk"] for r in rows) * len(pts) > MAX_EXACT_NODES:
            return None
        if kind == "design":
            return _exact_design(rows, pts, np.random.default_rng(seed + 1).standard_normal(pts.shape) / len(pts))
        out = _exact_fields(rows, pts, case["q"])
        if kind == "dropin":
            return out[case["q"]].reshape(-1, 3, 3) if case["q"] == "G" else out[case["q"]]
        return out
    prim, sec, i, j = _pair_rows(case, seed)
    if kind == "coaxial":
        return _exact_coaxial(prim, sec)
    pairs = zip(prim, sec) if i is None else ((prim[a], sec[b]) for a, b in zip(i, j))
    if sum(p["n_ang"] * p["n_thk"] * s["n_ang"] * s["n_thk"] * s["n_len"] for p, s in pairs) > MAX_EXACT_NODES:
        return None
    if kind == "pairs_grad":
        return _exact_pairs_grad(prim, sec)
    out = _exact_pairs(prim, sec, i, j)
    return {k: out.get(k) for w in case["what"] for k in dict(M=("M",), F=("F", "T"), D=("dM",))[w]}
