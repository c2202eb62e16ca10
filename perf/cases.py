"""The work that the performance of this framework is judged by: calls of its public entry
points (tau solves in every precision, batches, the request loop, reactive area density and the
reachable-pore mask) on seeded synthetic volumes of the sizes its workloads and tests use.

listed() gives fixed cases, draw() more of the same ranges, prepare() what a program holds
before the call, run() one call with its outputs, work() the bytes no implementation can do
without, and exact() the outputs of a plain FP64 solve in torch where one is quick enough.

Volumes are the library's ellipsoid volumes (semi-axes a, a r, a r, a = 12, solid fraction
0.5 .. 0.75), as in the benchmark, the batched and the serving workloads.  Plate-like bodies
(r > 1) are solved to 1e-9, as those workloads do; needle-like and compact ones (r <= 1) also to
the command line's default 1e-6 and to 1e-8.

A mixed solve's tau is kept in a single-precision table: the form stores its vectors in FP32
and is asked for a residual, not for digits.  The FP64 and FP32 forms follow fixed recurrences,
so their iteration counts are outputs too.
"""
import math

import numpy as np
import torch

from fast_amd import tau as T

A_SEMI = 12.0
CG, BICG = 1, 0
COEFFS = (1.0, 0.001)
DIRS = {"x": 0, "-x": 1, "y": 2, "-y": 3, "z": 4, "-z": 5, "xyz": None}


def listed():
    return [
        # the smallest volume of the request mix, one direction: launches and polling count
        {"name": "tau_mixed_64", "kind": "tau", "nx": 64, "ny": 64, "nz": 64, "r": 0.35, "solid": 0.65,
         "dir": "x", "precision": "mixed", "solver": "cg", "tol": 1e-6},
        # the benchmark's step: the three directions of a resident 256^3 volume, `fast tau -d xyz`
        {"name": "tau_mixed_256_xyz", "kind": "tau", "nx": 256, "ny": 256, "nz": 256, "r": 0.35, "solid": 0.65,
         "dir": "xyz", "precision": "mixed", "solver": "cg", "tol": 1e-6},
        # the largest volume of the request mix, needles, to 1e-8
        {"name": "tau_mixed_384", "kind": "tau", "nx": 384, "ny": 384, "nz": 384, "r": 0.1, "solid": 0.55,
         "dir": "z", "precision": "mixed", "solver": "cg", "tol": 1e-8},
        # volumes of uneven sizes and shapes in one batched solve
        {"name": "batch_mixed_24", "kind": "batch", "count": 24, "lo": 32, "hi": 192, "tol": 1e-9},
        # the command line's defaults (FP64 CG, 1e-6) on a small volume, with the concentration field
        {"name": "tau_fp64_cg_64_field", "kind": "tau", "nx": 64, "ny": 64, "nz": 64, "r": 0.5, "solid": 0.6,
         "dir": "x", "precision": "double", "solver": "cg", "tol": 1e-6, "field": True},
        # the same solver on an ordinary volume with odd edges
        {"name": "tau_fp64_cg_191", "kind": "tau", "nx": 191, "ny": 205, "nz": 177, "r": 0.35, "solid": 0.65,
         "dir": "y", "precision": "double", "solver": "cg", "tol": 1e-6},
        # `--solver bicgstab`, against the axis
        {"name": "tau_fp64_bicgstab_112", "kind": "tau", "nx": 112, "ny": 96, "nz": 130, "r": 0.35, "solid": 0.65,
         "dir": "-z", "precision": "double", "solver": "bicgstab", "tol": 1e-6},
        # `-p float`
        {"name": "tau_fp32_cg_128", "kind": "tau", "nx": 128, "ny": 128, "nz": 128, "r": 0.35, "solid": 0.65,
         "dir": "x", "precision": "float", "solver": "cg", "tol": 1e-5},
        # `fast alpha`, the whole-volume row of a resident volume
        {"name": "alpha_area_256", "kind": "area", "nx": 256, "ny": 256, "nz": 256, "r": 0.35, "solid": 0.65},
        # `fast alpha`, the six per-face rows of a volume that comes from the host
        {"name": "alpha_tensor_250", "kind": "tensor", "nx": 250, "ny": 233, "nz": 241, "r": 0.35, "solid": 0.65},
        # reachable-pore mask of a volume that comes from the host
        {"name": "reachable_192", "kind": "reach", "nx": 192, "ny": 192, "nz": 192, "r": 0.35, "solid": 0.65,
         "dir": "z"},
        # a burst of requests into the request loop
        {"name": "serve_burst_12", "kind": "serve", "count": 12, "lo": 64, "hi": 192, "tol": 1e-9},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _edges(rng, lo, hi):
    """Three edges around a log-uniform size, odd ones among them, none above hi."""
    e = _log(rng, lo, hi)
    return [max(lo // 2, min(hi, int(round(e * rng.uniform(0.75, 1.25))))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["tau", "tau", "tau", "tau", "batch", "area", "tensor", "reach", "serve"])
    c = {"kind": kind}
    if kind in ("batch", "serve"):
        c["count"] = rng.randint(4, 20) if kind == "batch" else rng.randint(4, 12)
        c["lo"], c["hi"] = rng.randint(24, 64), rng.randint(96, 176)
        c["tol"] = 1e-9
        return c
    if kind == "tau":
        form = rng.choice(["mixed", "mixed", "double", "bicgstab", "float"])
        hi = {"mixed": 352, "double": 208, "bicgstab": 160, "float": 192}[form]
        c["nx"], c["ny"], c["nz"] = _edges(rng, 48, hi)
        c["r"] = round(math.exp(rng.uniform(math.log(0.1), 0.0)), 3)
        c["solid"] = round(rng.uniform(0.5, 0.7), 3)
        c["dir"] = rng.choice(["x", "-x", "y", "-y", "z", "-z"])
        c["precision"] = "double" if form == "bicgstab" else form
        c["solver"] = "bicgstab" if form == "bicgstab" else "cg"
        c["tol"] = {"mixed": rng.choice([1e-6, 1e-8, 1e-9]), "double": 1e-6, "bicgstab": 1e-6, "float": 1e-5}[form]
        return c
    c["nx"], c["ny"], c["nz"] = _edges(rng, 48, 288)
    c["r"] = round(math.exp(rng.uniform(math.log(0.1), math.log(10.0))), 3)
    c["solid"] = round(rng.uniform(0.5, 0.75), 3)
    if kind == "reach":
        c["dir"] = rng.choice(["x", "y", "z"])
    return c


# ---- inputs --------------------------------------------------------------------------------
def _mask(case, seed):
    return T.generate_ellipsoids((case["nx"], case["ny"], case["nz"]), A_SEMI, case["r"], case["solid"], seed)


def _uneven(case, seed):
    """Masks and directions of a batch or burst: sizes, shapes and directions are those of the
    case, the volumes' contents come from the seed.  A batch's edges are independent per axis, a
    request's volume is a cube."""
    fixed = np.random.default_rng(1000 + case["count"])
    out = []
    for i in range(case["count"]):
        n = fixed.integers(case["lo"], case["hi"] + 1, size=3)
        if case["kind"] == "serve":
            n[:] = n[0]
        r = float(math.exp(fixed.uniform(math.log(0.1), math.log(10.0))))
        solid = float(fixed.uniform(0.5, 0.75))
        m = T.generate_ellipsoids(tuple(int(v) for v in n), A_SEMI, r, solid, 1000 * seed + i)
        out.append((m, (0, 2, 4)[i % 3]))
    return out


def _directions(case):
    return [0, 2, 4] if case["dir"] == "xyz" else [DIRS[case["dir"]]]


def _params(d, case):
    return T.make_params(d, BICG if case.get("solver") == "bicgstab" else CG, case.get("precision", "mixed"),
                         case["tol"], 40000, COEFFS)


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "mixed": case.get("precision", "mixed") == "mixed", "field": bool(case.get("field"))}
    if kind in ("batch", "serve"):
        items = _uneven(case, seed)
        s["params"] = [_params(d, case) for _, d in items]
        if kind == "batch":
            s["ctx"] = T.default_context()
            s["vols"] = [s["ctx"].volume(m) for m, _ in items]
        else:
            s["masks"] = [m for m, _ in items]
            s["ctx"] = T.Context(0)   # a request loop owns its context
            s["server"] = T.Server(s["ctx"], hbm_budget=4 << 30, iters_per_round=16)
        return s
    m = _mask(case, seed)
    if kind == "tau":
        s["ctx"] = T.default_context()
        s["vols"] = [s["ctx"].volume(m)] * len(_directions(case))
        s["params"] = [_params(d, case) for d in _directions(case)]
    elif kind == "area":
        s["vol"] = T.default_context().volume(m)
    else:
        s["mask"] = m
        s["dir"] = DIRS.get(case.get("dir", "z"))
    return s


def _table(results, mixed):
    tau = np.array([r.tau for r in results], dtype=np.float32 if mixed else np.float64)
    out = {"tau": tau, "porosity": np.array([r.porosity for r in results])}
    if not mixed:
        out["iterations"] = np.array([r.iterations for r in results])
    return out


def run(s):
    kind = s["kind"]
    if kind in ("tau", "batch"):
        if len(s["vols"]) == 1:
            res, field = s["vols"][0].solve(s["params"][0], conc=s["field"])
            out = _table([res], s["mixed"])
            if field is not None:
                out["field"] = field
            return out
        return _table(T.solve_batch(s["ctx"], s["vols"], s["params"]), s["mixed"])
    if kind == "serve":
        tickets = [s["server"].submit(m, p) for m, p in zip(s["masks"], s["params"])]
        got = {}
        while len(got) < len(tickets):
            ticket, res, _ = s["server"].wait()
            got[ticket] = res
        return _table([got[t] for t in tickets], True)
    if kind == "area":
        return s["vol"].area()
    if kind == "tensor":
        return T.getReactiveAreaDensityTensor(s["mask"])
    vol = T.default_context().volume(s["mask"])
    mask, labels = vol.reachable_mask(s["dir"])
    vol.close()
    return {"mask": mask, "labels": labels}


# ---- what cannot be done without -------------------------------------------------------------
def work(case):
    """Bytes: each mask byte read once; a solve forms its FP64 field once per direction; a
    reachable mask is written once."""
    if case["kind"] in ("batch", "serve"):
        n = [m.size for m, _ in _uneven(case, 1)]
        return {"bytes": 9.0 * sum(n), "flops": 0.0}
    n = float(case["nx"]) * case["ny"] * case["nz"]
    if case["kind"] == "tau":
        return {"bytes": n + 8.0 * n * len(_directions(case)), "flops": 0.0}
    return {"bytes": 2.0 * n if case["kind"] == "reach" else n, "flops": 0.0}


# ---- a plain FP64 solve ------------------------------------------------------------------------
def _solve64(mask, d, device):
    """tau and the concentration field of the converged solution: Jacobi CG in FP64 on the
    finite-volume system (arithmetic-mean face coefficients, half cells at the two faces of the
    flow axis, no flux through the others)."""
    solid = torch.from_numpy(mask).to(device) != 0
    one, low = (float(np.float32(v)) for v in COEFFS)
    axis = 2 - d // 2
    D = torch.where(solid, low, one).to(torch.float64)
    D = D.movedim(axis, 0)
    if d % 2:
        D = D.flip(0)
    D = D.contiguous()
    n = D.shape[0]
    face = [(D.narrow(a, 1, D.shape[a] - 1) + D.narrow(a, 0, D.shape[a] - 1)) * 0.5 for a in range(3)]
    ends = torch.zeros_like(D)
    ends[0] += 2 * D[0]
    ends[n - 1] += 2 * D[n - 1]
    diag = ends.clone()
    for a in range(3):
        m = D.shape[a] - 1
        diag.narrow(a, 0, m).add_(face[a])
        diag.narrow(a, 1, m).add_(face[a])

    def apply(p):
        y = ends * p
        for a in range(3):
            m = D.shape[a] - 1
            f = (p.narrow(a, 1, m) - p.narrow(a, 0, m)).mul_(face[a])
            y.narrow(a, 0, m).sub_(f)
            y.narrow(a, 1, m).add_(f)
        return y

    b = torch.zeros_like(D)
    b[0] = 2 * D[0]
    k = torch.arange(n, dtype=torch.float64, device=device)
    x = (1 - k / (n + 1)).reshape(n, 1, 1).expand_as(D).clone()
    r = b - apply(x)
    stop = 1e-24 * float((b * b).sum())
    z = r / diag
    p = z.clone()
    rz = (r * z).sum()
    for it in range(20000):
        q = apply(p)
        alpha = rz / (p * q).sum()
        x.addcmul_(alpha, p)
        r.addcmul_(-alpha, q)
        if it % 50 == 49 and float((r * r).sum()) <= stop:
            break
        z = r / diag
        new = (r * z).sum()
        p.mul_(new / rz).add_(z)
        rz = new
    flux = D[:-1] * (x[:-1] - x[1:])
    dc = (float(flux.sum()) + float((D[-1] * x[-1] / 0.5).sum())) / x.numel()
    porosity = float(np.float32(float((~solid).sum()) / solid.numel()))
    field = (x.flip(0) if d % 2 else x).movedim(0, axis)
    return porosity / (dc * n), porosity, field


def exact(case, seed):
    kind = case["kind"]
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "tau":
        if case["nx"] * case["ny"] * case["nz"] * len(_directions(case)) > 2.5e7:
            return None
        m = _mask(case, seed)
        items = [(m, d) for d in _directions(case)]
    elif kind in ("batch", "serve"):
        items = _uneven(case, seed)
        if sum(m.size for m, _ in items) > 1.5e7:
            return None
    else:
        return None
    got = [_solve64(m, d, device) for m, d in items]
    out = {"tau": np.array([g[0] for g in got]), "porosity": np.array([g[1] for g in got])}
    if case.get("precision", "mixed") != "mixed":
        out["iterations"] = None
    if case.get("field"):
        out["field"] = got[0][2].cpu().numpy()
    return out
