"""The work that programs have this package do, as cases that can be timed and checked.

A case is a dict of plain values; its "kind" says which public entry points it calls:

  coef3d    Context.coef_3d then coef_i_3d of a batch of domain arrays: a program that takes
            fields to coefficients and back (Base_spectral::coef / coef_i)
  residual  XctsSystem / DeviceSystem.residual(): F(u), once per Newton iteration and once
            per try of the line search
  jacobian  XctsSystem.jacobian(): the whole J of a system that fits a dense matrix
  columns   DeviceSystem.jvp_fill(): a range of columns of J, in fp64 or fp32
  vjp       DeviceSystem.vjp(): J^T w without J (the adjoint's gradient)
  newton    two do_newton() iterations from a guess, with the solver named
  lu        Context.lu_factor() and lu_solve() of one dense fp64 matrix
  refine    an fp64 system solved by low-precision factors: cast_f32, lu_factor("f32" or
            "bf16") and ir_solve() by flexible GMRES

listed() gives the sizes of this repository's own configurations (9x7x4 with 3 domains,
13x9x8 with 4, 17x13x12 with 5) and dense orders between them; draw() spreads over the
same ranges, odd sizes included.
"""
import functools
import math

import numpy as np
import torch

from kadath_frontera_amd import programs
from kadath_frontera_amd.device import Context
from kadath_frontera_amd.xcts import XctsSystem

# basis ids of include/base_spectral.hpp
CHEB, COSSIN, COS_EVEN, COS_ODD, SIN_EVEN, SIN_ODD = 1, 4, 6, 7, 9, 10
BOUNDS = [1.0, 2.0, 4.0, 8.0, 16.0]
N0, A, OME = 0.5, 1.0, 0.05  # lapse on the excision sphere, its radius, horizon rotation


def listed():
    return [
        # one field of one small domain: launch and synchronisation latency
        {"name": "coef3d_9x7x4_one", "kind": "coef3d", "nr": 9, "nt": 7, "np": 4, "batch": 1, "anti": False},
        # a full batch of Jacobian tangents at the production resolution
        {"name": "coef3d_17x13x12_4096", "kind": "coef3d", "nr": 17, "nt": 13, "np": 12, "batch": 4096, "anti": False},
        # the residual of the configuration that a desktop run starts with
        {"name": "residual_9x7x4", "kind": "residual", "nr": 9, "nt": 7, "np": 4, "domains": 3, "strings": False},
        # the residual of the production spinning hole, declared by equation strings
        {"name": "residual_17x13x12_strings", "kind": "residual", "nr": 17, "nt": 13, "np": 12, "domains": 5,
         "strings": True},
        # a whole small Jacobian (a program with its own linear algebra)
        {"name": "jacobian_9x7x4", "kind": "jacobian", "nr": 9, "nt": 7, "np": 4, "domains": 3, "batch": 512},
        # a tile of fp32 columns across several fields and domains of the production system
        {"name": "columns_17x13x12_f32", "kind": "columns", "nr": 17, "nt": 13, "np": 12, "domains": 5,
         "begin": 12345, "count": 5001, "dtype": "f32", "batch": 4096},
        # one adjoint product of an intermediate resolution
        {"name": "vjp_13x9x8", "kind": "vjp", "nr": 13, "nt": 9, "np": 8, "domains": 4, "batch": 1024},
        # Newton on the small configuration with the reference's algorithm (one fp64 LU)
        {"name": "newton_9x7x4_f64", "kind": "newton", "nr": 9, "nt": 7, "np": 4, "domains": 3, "solver": "f64",
         "batch": 512},
        # Newton on the production spinning hole with the fastest factor-every-step solver
        {"name": "newton_17x13x12_f64dd", "kind": "newton", "nr": 17, "nt": 13, "np": 12, "domains": 5,
         "solver": "f64-dd", "batch": 4096},
        # a small dense system: bound by the panel chain's launches
        {"name": "lu_1215", "kind": "lu", "n": 1215},
        # a large dense system of odd order
        {"name": "lu_8191", "kind": "lu", "n": 8191},
        # mixed precision: fp32 factors, fp64 refinement
        {"name": "refine_4321_f32", "kind": "refine", "n": 4321, "prec": "f32"},
    ]


def draw(rng):
    kind = rng.choice(["coef3d", "residual", "jacobian", "columns", "vjp", "newton", "lu", "refine"])
    if kind == "coef3d":
        nr, nt, npt = rng.randint(5, 33), rng.randint(5, 13), 4 * rng.randint(1, 4)
        most = 4096 * 17 * 13 * 12 // (nr * nt * npt)
        return {"kind": kind, "nr": nr, "nt": nt, "np": npt, "batch": _log_int(rng, 1, min(8192, most)),
                "anti": rng.random() < 0.5}
    if kind == "lu":
        return {"kind": kind, "n": _log_int(rng, 200, 8191)}
    if kind == "refine":
        return {"kind": kind, "n": _log_int(rng, 200, 4321), "prec": rng.choice(["f32", "f32", "bf16"])}
    # a dense J of the whole system (jacobian, newton) is kept below about 16000 unknowns
    whole = kind in ("jacobian", "newton")
    nr, nt = rng.randint(5, 13 if whole else 17), rng.randint(5, 9 if whole else 13)
    npt, nd = 4 * rng.randint(1, 2 if whole else 3), rng.randint(2, 4 if whole else 5)
    c = {"kind": kind, "nr": nr, "nt": nt, "np": npt, "domains": nd}
    if kind == "residual":
        c["strings"] = rng.random() < 0.5
        return c
    c["batch"] = rng.choice([256, 512, 1024]) if whole else rng.choice([512, 1024, 4096])
    if kind == "columns":
        n = _unknowns(c)
        c["count"] = _log_int(rng, 16, min(5001, n))
        c["begin"] = rng.randint(0, n - c["count"])
        c["dtype"] = rng.choice(["f64", "f32"])
    if kind == "newton":
        c["solver"] = rng.choice(["f64", "f64-dd", "f32-gmres"])
    return c


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _unknowns(c):
    """A lower bound of the unknowns of the 5-field system (exact sizes are the system's)."""
    return int(0.85 * 5 * c["domains"] * c["nr"] * (c["nt"] - 1) * c["np"])


# ---- spectral transforms in plain torch: the collocation points and basis functions ------
def _theta_bases(npt, anti):
    return [((COS_ODD, SIN_EVEN) if anti else (COS_EVEN, SIN_ODD))[(k // 2) % 2] for k in range(npt + 2)]


@functools.lru_cache(maxsize=None)
def _synthesis(base, n):
    """Values at the n collocation points (rows) of the basis functions (columns)."""
    if base == CHEB:
        x = -np.cos(np.pi * np.arange(n) / (n - 1))
        return np.cos(np.arange(n)[None] * np.arccos(x)[:, None])
    if base == COSSIN:
        p, k = 2 * np.pi * np.arange(n)[:, None] / n, np.arange(n + 2)
        s = np.where(k % 2 == 0, np.cos((k // 2) * p), np.sin((k // 2) * p))
        s[:, [1, n + 1]] = 0.0  # sin(0) and sin(n/2 phi)
        return s
    t, j = np.pi / 2 * np.arange(n)[:, None] / (n - 1), np.arange(n)
    s = {COS_EVEN: np.cos(2 * j * t), COS_ODD: np.cos((2 * j + 1) * t), SIN_EVEN: np.sin(2 * j * t),
         SIN_ODD: np.sin((2 * j + 1) * t)}[base]
    if base == SIN_EVEN:
        s[:, [0, n - 1]] = 0.0
    elif base != COS_EVEN:
        s[:, n - 1] = 0.0  # n - 1 functions on n points
    return s


@functools.lru_cache(maxsize=None)
def _analysis(base, n):
    s = _synthesis(base, n)
    keep = np.abs(s).max(axis=0) > 1e-9
    out = np.zeros(s.T.shape)
    out[keep] = np.linalg.pinv(s[:, keep])
    return out


def _along(m, x, axis):
    m = torch.tensor(m, dtype=torch.float64, device=x.device)
    return torch.movedim(torch.movedim(x, axis, -1) @ m.T.contiguous(), -1, axis)


def _theta(x, bt, matrix, nt):
    """A theta pass of (batch, phi coefficient, theta, r): the basis follows the phi index."""
    return torch.stack([_along(matrix(b, nt), x[:, k], 1) for k, b in enumerate(bt)], dim=1)


def _to_conf(cf, bt):
    npt, nt, nr = cf.shape[1] - 2, cf.shape[2], cf.shape[3]
    return _along(_synthesis(COSSIN, npt), _theta(_along(_synthesis(CHEB, nr), cf, 3), bt, _synthesis, nt), 1)


def _to_coef(conf, bt):
    npt, nt, nr = conf.shape[1:]
    return _along(_analysis(CHEB, nr), _theta(_along(_analysis(COSSIN, npt), conf, 1), bt, _analysis, nt), 3)


# ---- inputs ------------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _context():
    return Context(0)  # one per GPU, as a program holds it


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _coefs(case, seed):
    """Coefficients of smooth fields: U(-1, 1) 2^-(i+j+k), zero where the basis has no function."""
    nr, nt, npt = case["nr"], case["nt"], case["np"]
    g = _generator(seed)
    cf = 2 * torch.rand((case["batch"], npt + 2, nt, nr), dtype=torch.float64, device="cuda", generator=g) - 1
    i, j, k = (torch.arange(m, device="cuda", dtype=torch.float64) for m in (nr, nt, npt + 2))
    cf *= torch.exp2(-(i[None, None] + j[None, :, None] + (k // 2)[:, None, None]))
    live = torch.tensor(np.abs(_synthesis(COSSIN, npt)).max(axis=0) > 1e-9, device="cuda")
    cf *= live[:, None, None]
    for q, b in enumerate(_theta_bases(npt, case["anti"])):
        cf[:, q] *= torch.tensor(np.abs(_synthesis(b, nt)).max(axis=0) > 1e-9, device="cuda")[:, None]
    return cf


def _system(case):
    res, bounds = (case["nr"], case["nt"], case["np"]), BOUNDS[:case["domains"]]
    batch = case.get("batch", 256)
    strings = case["kind"] in ("columns", "vjp") or case.get("strings") or case.get("solver") in ("f64", "f32-gmres")
    if not strings:
        return XctsSystem(_context(), res, bounds, n0=N0, a=A, ome=OME, batch=batch, order=1)
    sd = programs.kerr(_context(), res, bounds, n0=N0, a=A, ome=OME)
    radius = {d: sd.coloc(d)[0] for d in range(1, len(bounds) + 1)}
    s = sd.build(order=1, batch=batch)
    for d, r in radius.items():  # the flat guess; infinity is a collocation point of the last domain
        s.set_field("P", d, 1.0 + A / r)
        s.set_field("N", d, np.ones_like(r))
        for f in ("bet^x", "bet^y", "bet^z"):
            s.set_field(f, d, np.zeros_like(r))
    return s


def _perturb(s, seed):
    """The flat guess plus a seeded 1e-3 perturbation of every coefficient."""
    X0 = s.perturbation(seed + 1)
    if isinstance(s, XctsSystem):
        s.set_guess(X0)
    else:
        s.add_unknowns(X0)


def _matrix(n, seed, shift=0.0):
    """Column-major dense matrix of normal entries (+ shift on the diagonal) and a right-hand side."""
    g = _generator(seed)
    At = torch.randn((n, n), dtype=torch.float64, device="cuda", generator=g)
    if shift:
        At.diagonal().add_(shift)
    return At, torch.randn(n, dtype=torch.float64, device="cuda", generator=g)


def _shift(case):
    # refinement needs factors that precondition: bf16 keeps 8 bits, so its system is well conditioned
    return (4.0 if case["prec"] == "bf16" else 0.5) * math.sqrt(case["n"])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "coef3d":
        bt = _theta_bases(case["np"], case["anti"])
        cf = _coefs(case, seed)
        conf = _to_conf(_coefs(case, seed + 7), bt).contiguous()
        base = ([CHEB] * ((case["np"] + 2) * case["nt"]), bt, COSSIN)
        return {"case": case, "conf": conf, "coef": cf, "base": base}
    if kind in ("lu", "refine"):
        At, b = _matrix(case["n"], seed, _shift(case) if kind == "refine" else 0.0)
        # the buffer that each solve factors in place, as a program that fills a matrix per step keeps it
        lo = torch.empty_like(At, dtype=torch.float32 if kind == "refine" else torch.float64)
        return {"case": case, "At": At, "b": b, "work": lo}
    s = _system(case)
    st = {"case": case, "system": s}
    _perturb(s, seed)
    if kind == "vjp":
        st["w"] = torch.randn(s.m, dtype=torch.float64, device="cuda", generator=_generator(seed))
    if kind == "newton":
        st["guess"] = {(f, d): s.coef(f, d).copy() for f in range(5) for d in range(1, case["domains"] + 1)}
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "coef3d":
        ctx, base = _context(), state["base"]
        return ctx.coef_3d(state["conf"], *base), ctx.coef_i_3d(state["coef"], *base)
    if kind == "lu":
        ctx, W = _context(), state["work"]
        W.copy_(state["At"])
        ipiv, perm, info = ctx.lu_factor("f64", W.T)
        x = ctx.lu_solve("f64", W.T, perm, state["b"].clone())
        return {"x": x, "lu": W, "ipiv": ipiv, "perm": perm, "info": info}
    if kind == "refine":
        # the factors' last bits follow the order of 32-bit sums; what the path gives is x
        ctx, A64, lo = _context(), state["At"].T, state["work"].T
        ctx.cast_f32(A64, lo)
        _, perm, info = ctx.lu_factor(case["prec"], lo)
        x, _, _, done = ctx.ir_solve(A64, case["prec"], lo, perm, state["b"], mode=1)
        return {"x": x, "info": info, "done": done}
    s = state["system"]
    if kind == "residual":
        return s.residual()
    if kind == "jacobian":
        return s.jacobian()
    if kind == "columns":
        return s.jvp_fill(case["begin"], case["count"], dtype=torch.float32 if case["dtype"] == "f32" else torch.float64)
    if kind == "vjp":
        return s.vjp(state["w"])
    # newton: two iterations of a new solve from the guess, and the fields they reach
    for (f, d), cf in state["guess"].items():
        s.set_coef(f, d, cf)
    s.set_option(drop_factors=True)
    errors = [s.do_newton(1e-10, case["solver"])[1] for _ in range(2)]
    return {"F_max": np.array(errors),
            "fields": np.concatenate([s.coef(f, d).ravel() for f in range(5) for d in range(1, case["domains"] + 1)])}


def work(case):
    kind = case["kind"]
    if kind == "coef3d":
        # conf and coef arrays once in each direction; fast transforms of every line
        nr, nt, npt, nb = case["nr"], case["nt"], case["np"], case["batch"]
        conf, coef = nr * nt * npt, nr * nt * (npt + 2)
        return {"bytes": 16.0 * nb * (conf + coef), "flops": 10.0 * nb * coef * math.log2(coef)}
    if kind in ("lu", "refine"):
        n = float(case["n"])
        return {"bytes": 16.0 * n * n, "flops": 2.0 / 3.0 * n ** 3 + 2.0 * n * n}
    nd, npts = case["domains"], case["nr"] * case["nt"] * (case["np"] + 2)
    n, fields = _unknowns(case) / 0.85, 5 * nd * npts
    # a residual takes the first and second derivatives of five fields: 9 derivatives by 1-D
    # operators of about log2 cost per point, and the pointwise terms
    residual = {"bytes": 8.0 * (fields + n), "flops": 9.0 * fields * (5.0 * math.log2(npts) + 10.0)}
    if kind == "residual":
        return residual
    if kind == "jacobian":
        return {"bytes": 8.0 * (fields + n * n), "flops": residual["flops"]}
    if kind == "columns":
        return {"bytes": 8.0 * fields + (4.0 if case["dtype"] == "f32" else 8.0) * n * case["count"],
                "flops": residual["flops"]}
    if kind == "vjp":  # one reverse pass is a few residuals
        return {"bytes": 8.0 * (fields + 2.0 * n), "flops": 3.0 * residual["flops"]}
    # newton: J written and read once; the factors of J, or of its domain blocks
    nb = n / nd if case["solver"] == "f64-dd" else n
    blocks = nd if case["solver"] == "f64-dd" else 1
    return {"bytes": 2.0 * 2.0 * 8.0 * blocks * nb * nb, "flops": 2.0 * blocks * 2.0 / 3.0 * nb ** 3}


def tolerance(case):
    """About four times the difference seen between two evaluations with sums in another order."""
    if case.get("dtype") == "f32":
        return {"rel": 1e-7, "max": 2.5e-7}  # fp32 columns against rounded fp64 ones: 2.4e-8, 5.8e-8
    return TOLERANCE[case["kind"]]


TOLERANCE = {
    # line matrices against the basis functions' products: 3e-15
    "coef3d": {"rel": 2e-14, "max": 5e-13},
    # fp64 transforms by fast algorithms instead of line matrices: 1.8e-12 at 9x7x4, 1.2e-10 (4e-9
    # of the rms at most) at 17x13x12, where second derivatives amplify the coefficients' last bits
    "residual": {"rel": 5e-10, "max": 1.6e-8},
    # the same: 1.5e-15, 1.5e-13 at 9x7x4; two traces of the equations at 13x9x8: 5.6e-14 at most
    "jacobian": {"rel": 1e-13, "max": 1e-11},
    "columns": {"rel": 1e-13, "max": 1e-11},
    "vjp": {"rel": 1e-13, "max": 1e-11},
    # one LU of J against the domain-decomposed solve: fields 1.1e-10, and 2.5e-8 in the largest
    # |F| after the first step (it holds the directions that J nearly maps to zero)
    "newton": {"rel": 1e-7, "max": 4e-7},
    # against LAPACK: factors 7e-13, x 1.3e-11 at n = 8191; the condition of a random matrix
    # exceeds its median 50 times in a few per cent of the seeds
    "lu": {"rel": 1e-9, "max": 1e-8},
    # x of a residual at 1e-13 ||b||: 1e-12 at n = 4321, 1e-8 seen where the matrix is worse conditioned
    "refine": {"rel": 1e-7, "max": 1e-6},
}


def exact(case, seed):
    """Plain torch in 64 bits: the transforms from their basis functions, the dense systems by
    torch.linalg.  The Newton system's rows (tau conditions of traced equations) have no such
    plain form short of a second implementation of the method."""
    kind = case["kind"]
    if kind == "coef3d":
        bt = _theta_bases(case["np"], case["anti"])
        return _to_coef(_to_conf(_coefs(case, seed + 7), bt), bt), _to_conf(_coefs(case, seed), bt)
    if kind in ("lu", "refine"):
        At, b = _matrix(case["n"], seed, _shift(case) if kind == "refine" else 0.0)
        # LAPACK on the host: its pivots are the first largest entries, as lu_factor's
        LU, piv = torch.linalg.lu_factor(At.T.cpu())
        x = torch.linalg.lu_solve(LU, piv, b.cpu()[:, None])[:, 0]
        if kind == "refine":
            return {"x": x, "info": None, "done": None}
        return {"x": x, "lu": LU.T.contiguous(), "ipiv": None, "perm": None, "info": None}
    return None
