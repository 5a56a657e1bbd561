"""What the solve path is timed on: one call of a public entry point per case.

The cases are the calls a user of the library makes, on the seeded synthetic
LDU systems of unap_amd.meshgen (boxes of hexahedral cells, randomly
relabelled): A x, whole solves with every preconditioner family in FP64 and
with its FP32 counterpart, and batches of independent systems.  A state is what
a program holds before the call: the matrix, the preconditioner and its
hierarchy, the solver and the vectors, all in device memory.  Every solve
starts from x = 0 and returns x.
"""
import math
import time

import numpy as np
import torch

from unap_amd import hip, meshgen

# Multigrid parameters by name: the reference's Gauss-Seidel and Chebyshev
# cycles (every pairwise level, coarsest level by PCG + DIC), and the FP32
# hierarchies that the flexible CG runs (fixed cycle, dense coarsest solve).
_GS64 = dict(smoother=1, n_cells_coarsest=500, n_vcycles=1)
_CHEBY64 = dict(smoother=2, n_cells_coarsest=500, n_vcycles=1, n_post_sweeps=4, n_finest_sweeps=4)
_GS32 = dict(precision=32, smoother=1, n_cells_coarsest=4000, n_vcycles=1, cycle=1, pair_steps=4, level_sweep_growth=0)
_CHEBY32 = dict(precision=32, smoother=2, n_cells_coarsest=4000, n_vcycles=1, n_post_sweeps=4, n_finest_sweeps=4,
                cycle=1, pair_steps=7, level_sweep_growth=0, scaling=0, cheby_eig_ratio=3.0,
                cheby_eig_ratio_finest=12.0, cheby_boost=1.0)

# method -> (solver, preconditioner, its precision or multigrid parameters)
_METHODS = {
    "pcg_dic": ("PCG", "DIC", None),
    "fcg_dic32": ("FCG", "DIC", dict(precision=32)),
    "bicg_dilu": ("PBiCGStab", "DILU", None),
    "fbicg_dilu32": ("FBiCGStab", "DILU", dict(precision=32)),
    "pcg_amg_gs": ("PCG", "AMG", _GS64),
    "fcg_amg32_gs": ("FCG", "AMG", _GS32),
    "pcg_amg_cheby": ("PCG", "AMG", _CHEBY64),
    "fcg_amg32_cheby": ("FCG", "AMG", _CHEBY32),
    "mg_gs": ("MG", None, dict(smoother=1, n_cells_coarsest=50, n_vcycles=1)),
}


def _case(method, system, nx, ny, nz, rel_tol=1e-8):
    return {"method": method, "system": system, "nx": nx, "ny": ny, "nz": nz, "rel_tol": rel_tol}


def listed():
    return [
        # A x on the smallest mesh of the drop-in configurations: a caller's
        # own Krylov loop on a small domain, where launches and waits count.
        dict(_case("amul", "poisson", 32, 32, 32), name="amul_32"),
        # A x on a large asymmetric mesh with no round edge, beyond every cache.
        dict(_case("amul", "convdiff", 167, 160, 153), name="amul_ragged"),
        # The small drop-in solve: constant Poisson 32^3, to 1e-6.
        dict(_case("pcg_dic", "poisson", 32, 32, 32, 1e-6), name="pcg_dic_32"),
        # The symmetric pressure-like solve without multigrid, FP32 sweeps, on an odd box.
        dict(_case("fcg_dic32", "logunif3", 71, 50, 63, 1e-6), name="fcg_dic32_ragged"),
        # The transport solve: 128^3 convection-diffusion, FP64.
        dict(_case("bicg_dilu", "convdiff", 128, 128, 128), name="bicg_dilu_128"),
        # The same kind of system, mid-sized and odd, with FP32 sweeps.
        dict(_case("fbicg_dilu32", "convdiff", 97, 64, 75), name="fbicg_dilu32_ragged"),
        # The pressure solve as the reference configures it: 128^3, Gauss-Seidel cycles in FP64.
        dict(_case("pcg_amg_gs", "logunif3", 128, 128, 128), name="pcg_amg_gs_128"),
        # The same solve with the FP32 hierarchy, on an odd box.
        dict(_case("fcg_amg32_gs", "logunif3", 121, 96, 107), name="fcg_amg32_gs_ragged"),
        # Multigrid as the solver itself, small.
        dict(_case("mg_gs", "logunif3", 48, 41, 45, 1e-6), name="mg_gs_small"),
        # The pressure solve with the reference's Chebyshev cycles in FP64.
        dict(_case("pcg_amg_cheby", "logunif3", 120, 120, 120, 1e-6), name="pcg_amg_cheby_120"),
        # The largest solve: 256^3, FP32 Chebyshev cycles inside the FP64 flexible CG.
        dict(_case("fcg_amg32_cheby", "logunif4", 256, 256, 256), name="fcg_amg32_cheby_256"),
        # Many small domains at once: uneven boxes, 60% symmetric, one launch.
        {"method": "batch", "count": 96, "lo": 8, "hi": 48, "rel_tol": 1e-8, "name": "batch_96"},
    ]


def _edges(rng, cells, spread=1.6):
    """Three edges whose product is about `cells`, each up to `spread` off the cube's."""
    e = cells ** (1.0 / 3.0)
    a, b = (math.exp(rng.uniform(-1, 1) * math.log(spread)) for _ in range(2))
    return [max(8, round(v)) for v in (e * a, e * b, e / math.sqrt(a * b))]


# method -> the systems it is used on, its range of cells, its tolerances
_RANGES = {
    "amul": (("poisson", "logunif3", "convdiff"), 4e3, 4e6, (1e-8,)),
    "pcg_dic": (("poisson", "logunif3"), 4e3, 3e5, (1e-6,)),
    "fcg_dic32": (("poisson", "logunif3"), 4e3, 3e5, (1e-6,)),
    "bicg_dilu": (("convdiff",), 4e3, 2e6, (1e-6, 1e-8)),
    "fbicg_dilu32": (("convdiff",), 4e3, 2e6, (1e-6, 1e-8)),
    "pcg_amg_gs": (("poisson", "logunif3"), 2e4, 1.5e6, (1e-6,)),
    "fcg_amg32_gs": (("poisson", "logunif3"), 2e5, 2e6, (1e-6, 1e-8)),
    "mg_gs": (("poisson", "logunif3"), 2e4, 2e5, (1e-6,)),
    "pcg_amg_cheby": (("poisson", "logunif3"), 2e4, 1.5e6, (1e-6,)),
    "fcg_amg32_cheby": (("logunif3", "logunif4"), 5e5, 8e6, (1e-6, 1e-8)),
}


def draw(rng):
    method = rng.choice(sorted(_RANGES) + ["batch"])
    if method == "batch":
        lo = rng.randint(8, 12)
        return {"method": "batch", "count": round(math.exp(rng.uniform(math.log(12), math.log(160)))), "lo": lo,
                "hi": rng.randint(lo + 4, 44), "rel_tol": 1e-8}
    systems, least, most, tols = _RANGES[method]
    cells = math.exp(rng.uniform(math.log(least), math.log(most)))
    return _case(method, rng.choice(systems), *_edges(rng, cells), rng.choice(tols))


def _system(case, seed):
    """The box system of the case: Poisson with unit or log-uniform
    coefficients, or upwind convection-diffusion up to Peclet 5."""
    dims = case["nx"], case["ny"], case["nz"]
    kind, p0, shift = {
        "poisson": (meshgen.POISSON_CONST, 0.0, 1e-6),
        "logunif3": (meshgen.POISSON_LOGUNIF, -3.0, 1e-6),
        "logunif4": (meshgen.POISSON_LOGUNIF, -4.0, 1e-6),
        "convdiff": (meshgen.CONVDIFF, 5.0, 1e-3),
    }[case["system"]]
    return meshgen.box_system(*dims, kind, p0, 0.0, shift, seed)


def _batch_dims(case):
    """(nx, ny, nz, kind) of the batch's systems."""
    return [s[:4] for s in meshgen.batch_specs(case["count"], case["lo"], case["hi"])]


def _batch(case, seed):
    return [meshgen.batch_system((*d, seed * 1000003 + i)) for i, d in enumerate(_batch_dims(case))]


def _device(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def prepare(case, seed):
    if case["method"] == "batch":
        systems = _batch(case, seed)
        B = hip.Batch(systems, ["PCG" if s.symmetric else "PBiCGStab" for s in systems])
        B.set_config(1024, 2, 256)  # a program's fixed shape, so that no solve is spent on tuning
        b = _device(np.concatenate([s.b for s in systems]))
        return {"batch": B, "b": b, "x": torch.zeros_like(b), "rel_tol": case["rel_tol"]}
    s = _system(case, seed)
    A = hip.LduMatrix.from_system(s)
    b = _device(s.b)
    x = torch.zeros_like(b)
    if case["method"] == "amul":
        torch.cuda.synchronize()
        A.spmv(b, out=x)  # the matrix is laid out on the device by its first use
        return {"A": A, "b": b, "x": x}
    kind, pre, prm = _METHODS[case["method"]]
    limits = dict(rel_tol=case["rel_tol"], max_iter=1000)
    if kind == "MG":
        S = hip.Solver("MG", mg=hip.amg_params(**prm), **limits)
        S.solve(A, b, x=x)  # builds the hierarchy, which the solver keeps
    else:
        amg = None if prm is None else hip.amg_params(**prm)
        S = hip.Solver(kind, hip.Precond(A, pre, amg=amg), **limits)
    return {"A": A, "b": b, "x": x, "solver": S}


def run(state):
    x, b = state["x"], state["b"]
    if "batch" in state:
        x.zero_()
        state["batch"].solve(b, x=x, rel_tol=state["rel_tol"])
    elif "solver" in state:
        x.zero_()
        state["solver"].solve(state["A"], b, x=x)
    else:
        state["A"].spmv(b, out=x)
    return x


def work(case):
    """The matrix (coefficients, addresses of the faces) and the right-hand
    side read once, the result written once; a multiply and an add for each
    coefficient and vector element.  A solve needs this much for any one pass
    over its system, however many iterations it takes."""
    if case["method"] == "batch":
        sizes = [(x * y * z, 3 * x * y * z - x * y - y * z - z * x, k == meshgen.CONVDIFF)
                 for x, y, z, k in _batch_dims(case)]
    else:
        x, y, z = case["nx"], case["ny"], case["nz"]
        sizes = [(x * y * z, 3 * x * y * z - x * y - y * z - z * x, case["system"] == "convdiff")]
    return {"bytes": float(sum(24 * n + (24 if asym else 16) * f for n, f, asym in sizes)),
            "flops": float(sum(2 * n + 4 * f for n, f, _ in sizes))}


# ------------------------------------------------------------- 64-bit values
def _operator(n, l, u, lower, diag, upper):
    """x -> A x in float64, from rows of coefficients padded to the longest row."""
    l, u, lower, diag, upper = (_device(v) for v in (l, u, lower, diag, upper))
    rows, order = torch.sort(torch.cat([l, u]), stable=True)
    cols, vals = torch.cat([u, l])[order], torch.cat([upper, lower])[order]
    count = torch.bincount(rows, minlength=n)
    at = torch.arange(rows.numel(), device=rows.device) - (torch.cumsum(count, 0) - count)[rows]
    width = int(count.max())
    col = torch.arange(n, device=rows.device).repeat(width, 1)
    val = torch.zeros(width, n, dtype=torch.float64, device=rows.device)
    col[at, rows], val[at, rows] = cols, vals

    def apply(x):
        y = diag * x
        for k in range(width):
            y = torch.addcmul(y, val[k], x[col[k]])
        return y

    return apply, diag


def _solve64(apply, diag, b, symmetric, limit_s=15.0):
    """A x = b to the accuracy of float64, by diagonally preconditioned CG or
    BiCGStab restarted from the true residual; None when that takes too long."""
    began, x, goal, best = time.perf_counter(), torch.zeros_like(b), float(b.norm()), None
    for _ in range(8):
        r = b - apply(x)
        size = float(r.norm())
        if best is not None and size > 0.5 * best:
            break
        best = size if best is None else min(best, size)
        if size <= 1e-15 * goal:
            break
        e = torch.zeros_like(b)
        if symmetric:
            z = r / diag
            p, rz = z.clone(), torch.dot(r, z)
        else:
            r0, p, rho = r.clone(), r.clone(), torch.dot(r, r)
        for it in range(100000):
            if symmetric:
                q = apply(p)
                a = rz / torch.dot(p, q)
                e, r = e + a * p, r - a * q
                z = r / diag
                new = torch.dot(r, z)
                p, rz = z + (new / rz) * p, new
            else:
                y = p / diag
                v = apply(y)
                a = rho / torch.dot(r0, v)
                s = r - a * v
                z = s / diag
                t = apply(z)
                w = torch.dot(t, s) / torch.dot(t, t)
                e, r = e + a * y + w * z, s - w * t
                new = torch.dot(r0, r)
                p, rho = r + (new / rho) * (a / w) * (p - w * v), new
            if it % 25 == 24:
                now = float(r.norm())
                if time.perf_counter() - began > limit_s:
                    return None
                if not math.isfinite(now) or now <= 1e-10 * size:
                    break
        if not bool(torch.isfinite(e).all()):
            return None
        x = x + e
    return x if best is not None and best <= 1e-11 * goal else None


def exact(case, seed):
    """A x, or the solution of A x = b, in float64 by torch."""
    if case["method"] == "batch":
        group, systems = {}, _batch(case, seed)
        for symmetric in (True, False):
            ids = [i for i, s in enumerate(systems) if s.symmetric == symmetric]
            if not ids:
                continue
            # the systems of one kind as one block-diagonal system
            off = np.concatenate([[0], np.cumsum([systems[i].n for i in ids])])
            cat = {k: np.concatenate([getattr(systems[i], k) + (off[j] if k in "lu" else 0) for j, i in enumerate(ids)])
                   for k in ("l", "u", "diag", "upper", "b")}
            lower = np.concatenate([systems[i].lower_or_upper() for i in ids])
            apply, diag = _operator(int(off[-1]), cat["l"], cat["u"], lower, cat["diag"], cat["upper"])
            x = _solve64(apply, diag, _device(cat["b"]), symmetric)
            if x is None:
                return None
            group.update({i: x[off[j]:off[j + 1]] for j, i in enumerate(ids)})
        return torch.cat([group[i] for i in range(len(systems))])
    if case["method"] != "amul" and case["nx"] * case["ny"] * case["nz"] > 3e6:
        return None
    s = _system(case, seed)
    apply, diag = _operator(s.n, s.l, s.u, s.lower_or_upper(), s.diag, s.upper)
    b = _device(s.b)
    return apply(b) if case["method"] == "amul" else _solve64(apply, diag, b, s.symmetric)
