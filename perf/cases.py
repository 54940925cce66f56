"""Performance cases: what programs built on fmca_amd spend their time in.

Every case is one call (or one training step, or one solve) through a public
entry point, on synthetic points and right-hand sides made from a seed.

  listed()             the fixed cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  inputs on the GPU (host arrays where the entry point takes
                       host arrays) and the plan a program keeps
  run(state)           one pass, its outputs whole
  work(case)           bytes and operations the path cannot do without
  tolerance(case)      distance of another correct implementation
  exact(case, seed)    the same outputs from the dense kernel matrix in 64 bits

Fields of a case:
  kind      action    H2kernelActor.action_device (action_transpose_device)
            assembled action_device of an actor whose blocks are stored (assemble)
            oneshot   H2Matrix(...).action on host arrays, plan included
            evaluate  MultipoleFunctionEvaluator.evaluate on host arrays
            step      autograd.h2_matvec forward and backward
            solve     H2kernelActor.cg, GCR with FP64 residual replacement
  dim, n, m points, sources, targets (m = 0: the targets are the sources)
  points    "uniform" in the unit cube, or "mixture" of 16 Gaussians
  ktype, l  kernel and lengthscale
  interp    "tensor_product" or "total_degree", with deg and eta
  nrhs      right-hand sides
  precision "FP64", "FP32" or "FP32_BF16"
  transpose (action) apply the transpose
  wrt       (step) "al": coefficients and lengthscale; "alp": and the points
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import fmca_amd
from fmca_amd.autograd import H2Spec, h2_matvec

PRECISIONS = {"FP64": fmca_amd.FP64, "FP32": fmca_amd.FP32, "FP32_BF16": fmca_amd.FP32_BF16}


def _case(name, kind, **kw):
    c = {"name": name, "kind": kind, "dim": 3, "n": 0, "m": 0, "points": "uniform",
         "ktype": "MATERN32", "l": 0.5, "interp": "tensor_product", "deg": 4, "eta": 0.8,
         "nrhs": 1, "precision": "FP64", "transpose": False, "wrt": ""}
    c.update(kw)
    return c


def listed():
    return [
        # the smallest calls: one prediction vector on a few thousand points
        # (latency, launches and idle compute units)
        _case("small_one_rhs", "action", n=10_000, ktype="EXPONENTIAL", deg=3),
        # a small batch of columns in single precision
        _case("small_batch", "action", n=4_000, deg=3, nrhs=16, precision="FP32"),
        # the Python binding as a notebook uses it: host arrays in and out,
        # points seen for the first time, total-degree moments
        _case("notebook_call", "oneshot", dim=2, n=10_000, ktype="EXPONENTIAL", l=1.0,
              interp="total_degree", nrhs=10),
        # out-of-sample evaluation of an interpolant at its default (every
        # block dense): odd sizes, more sources than targets
        _case("interpolant_values", "evaluate", n=20_011, m=5_003, ktype="MATERN52", l=0.3,
              interp="total_degree", deg=3, eta=0.0, nrhs=3),
        # a handful of right-hand sides on a ragged mid-size set
        _case("ragged_few_rhs", "action", n=123_457, ktype="MATERN52", l=0.3, deg=3, nrhs=5,
              precision="FP32"),
        # stored blocks, applied again and again
        _case("stored_blocks", "assembled", n=100_000, nrhs=32),
        # clustered data, many right-hand sides, uneven interaction lists
        _case("clustered_many_rhs", "action", n=400_000, points="mixture", ktype="GAUSSIAN",
              l=0.1, nrhs=64, precision="FP32_BF16"),
        # learning coefficients, lengthscale and point positions in the plane
        _case("train_plane", "step", dim=2, n=200_000, l=0.3, deg=5, nrhs=8, wrt="alp"),
        # learning coefficients and lengthscale on a large set in 3-D
        _case("train_space", "step", n=1_000_000, ktype="EXPONENTIAL", l=0.25, nrhs=16,
              precision="FP32", wrt="al"),
        # one vector through a large matrix (power iterations, residual checks)
        _case("large_one_rhs", "action", n=1_000_000, precision="FP32"),
        # the plain double-precision product on a large set with a block of columns
        _case("large_block_fp64", "action", n=1_000_000, nrhs=32),
        # the largest: a block of systems to a 1e-8 residual (its iterations are
        # FP32_BF16 actions of 32 columns)
        _case("large_solve", "solve", n=1_000_000, nrhs=32, precision="FP32_BF16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["action"] * 6 + ["assembled", "oneshot", "evaluate", "solve"]
                      + ["step"] * 2)
    dim = rng.choice([3, 3, 3, 2, 2, 1]) if kind in ("action", "oneshot") else rng.choice([3, 2])
    c = _case("", kind, dim=dim)
    del c["name"]
    c["ktype"] = rng.choice(["EXPONENTIAL", "MATERN32", "MATERN52", "GAUSSIAN"])
    c["l"] = round(rng.uniform(0.1, 1.0), 3)
    c["interp"] = rng.choice(["tensor_product", "tensor_product", "total_degree"])
    c["deg"] = rng.randint(2, 5)
    c["precision"] = rng.choice(sorted(PRECISIONS))
    c["nrhs"] = rng.choice([1, 1, 2, 3, 5, 7, 8, 10, 16, 16, 17, 24, 32, 32, 48, 64])
    if kind == "action":
        c["n"] = _log(rng, 2_000, 1_000_000)
        c["eta"] = rng.choice([0.8, 0.8, 0.5])
        if rng.random() < 0.3:
            c["m"] = _log(rng, 1_000, c["n"])
            c["transpose"] = rng.random() < 0.5
        if rng.random() < 0.2:
            c["ktype"] = rng.choice(["MATERN72", "MATERN92", "INVMULTIQUADRIC"])
        if rng.random() < 0.25:
            c["points"] = "mixture"
    elif kind == "assembled":
        c["n"] = _log(rng, 3_000, 120_000)
        c["deg"] = rng.randint(2, 4)
        c["precision"] = rng.choice(["FP64", "FP32"])
    elif kind == "oneshot":
        c["n"] = _log(rng, 1_000, 200_000)
        c["nrhs"] = rng.choice([1, 3, 10, 16, 32])
        c["precision"] = "FP64"
        c["deg"] = rng.randint(2, 4)
    elif kind == "evaluate":
        c["n"] = _log(rng, 2_000, 60_000)
        c["m"] = _log(rng, 1_000, 20_000)
        c["eta"] = rng.choice([0.0, 0.8])
        c["interp"] = "total_degree"
        c["deg"] = rng.randint(2, 4)
        c["nrhs"] = rng.choice([1, 1, 2, 3, 8])
        c["precision"] = "FP64"
    elif kind == "step":
        c["n"] = _log(rng, 3_000, 400_000)
        c["nrhs"] = rng.choice([1, 2, 4, 8, 8, 11, 16])
        c["deg"] = rng.randint(3, 5)
        c["interp"] = "tensor_product"
        c["precision"] = rng.choice(["FP64", "FP32"])
        c["ktype"] = rng.choice(["EXPONENTIAL", "MATERN32", "MATERN52", "GAUSSIAN"])
        c["l"] = round(rng.uniform(0.2, 0.6), 3)
        c["wrt"] = rng.choice(["al", "alp"])
        if rng.random() < 0.25:
            c["m"] = _log(rng, 2_000, c["n"])
    else:
        c["n"] = _log(rng, 5_000, 300_000)
        c["ktype"] = rng.choice(["EXPONENTIAL", "MATERN32"])
        c["l"] = round(rng.uniform(0.2, 0.6), 3)
        c["interp"] = "tensor_product"
        c["deg"] = 4
        c["nrhs"] = rng.choice([1, 4, 8, 16, 32])
        c["precision"] = rng.choice(["FP64", "FP32", "FP32_BF16", "FP32_BF16"])
    # no more columns than keep the arrays at the largest case's size
    while c["n"] * c["nrhs"] > 32_000_000:
        c["nrhs"] = max(1, c["nrhs"] // 2)
    return c


# ---------------------------------------------------------------------------
# inputs

def _cloud(case, n, rng):
    """n points as a (dim, n) Fortran-ordered array."""
    d = case["dim"]
    if case["points"] == "mixture":
        centres = rng.random((16, d))
        which = rng.integers(0, 16, n)
        return np.asfortranarray(centres[which].T + 0.02 * rng.standard_normal((d, n)))
    return np.asfortranarray(rng.random((d, n)))


def _points(case, seed):
    """(sources, targets); targets is None where they are the sources."""
    rng = np.random.default_rng(seed)
    P = _cloud(case, case["n"], rng)
    if case["kind"] == "oneshot":  # [-1, 1]^dim
        P = np.asfortranarray(2.0 * P - 1.0)
    return P, (_cloud(case, case["m"], rng) if case["m"] else None)


def _normal(rows, nrhs, seed):
    """N(0, 1) columns, column-major on the GPU as the device entry points take them."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn((nrhs, rows), generator=g, dtype=torch.float64, device="cuda").t()


def _rhs(case, seed):
    return _normal(case["m"] if case["transpose"] else case["n"], case["nrhs"], seed + 1)


def _host_rhs(case, seed):
    return np.asfortranarray(
        np.random.default_rng(seed + 1).standard_normal((case["n"], case["nrhs"])))


def _ridge(case):
    return 1e-4 * case["n"]


def prepare(case, seed):
    P, T = _points(case, seed)
    K = fmca_amd.CovarianceKernel(case["ktype"], case["l"])
    s = {"case": case, "precision": PRECISIONS[case["precision"]], "kernel": K}
    kind = case["kind"]
    if kind == "oneshot":
        s.update(P=P, x=_host_rhs(case, seed))
        return s
    if kind == "evaluate":
        ev = fmca_amd.MultipoleFunctionEvaluator(K, P, T, case["eta"], case["deg"])
        s.update(ev=ev, P=P, T=T, x=_host_rhs(case, seed))
        return s
    if kind == "step":
        pts = torch.from_numpy(P).cuda()
        tgt = None if T is None else torch.from_numpy(T).cuda()
        l = torch.tensor(case["l"], dtype=torch.float64, requires_grad=True)
        spec = H2Spec(case["ktype"], deg=case["deg"], eta=case["eta"],
                      precision=s["precision"], interpolator=case["interp"])
        alpha = _rhs(case, seed)
        h2_matvec(alpha[:, :1].contiguous(), l.detach(), pts, spec, tgt)  # the plan
        if "p" in case["wrt"]:
            pts.requires_grad_(True)
            if tgt is not None:
                tgt.requires_grad_(True)
        s.update(points=pts, targets=tgt, l=l, spec=spec, alpha=alpha.requires_grad_(True),
                 G=_normal(case["m"] or case["n"], case["nrhs"], seed + 2))
        return s
    H = fmca_amd.H2kernelActor(K, P if T is None else T, P, case["deg"], case["eta"],
                               case["interp"])
    H.upload()
    if kind == "assembled":
        H.assemble(s["precision"])
    s.update(H=H, x=_rhs(case, seed))
    if kind == "solve":
        s.update(x0=torch.zeros_like(s["x"]))
    return s


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "oneshot":
        H = fmca_amd.H2Matrix(state["kernel"], state["P"], state["P"], c["deg"], c["eta"],
                              interpolator=c["interp"])
        return H.action(state["x"])
    if kind == "evaluate":
        return state["ev"].evaluate(state["P"], state["T"], state["x"])
    if kind == "step":
        y = h2_matvec(state["alpha"], state["l"], state["points"], state["spec"],
                      state["targets"])
        wrt = [state["alpha"], state["l"]]
        if "p" in c["wrt"]:
            wrt += [state["points"]] + ([] if state["targets"] is None else [state["targets"]])
        return [y.detach(), *torch.autograd.grad(y, wrt, state["G"])]
    if kind == "solve":
        return state["H"].cg(state["x"], x0=state["x0"], ridge=_ridge(c), tol=1e-8,
                             precision=state["precision"], refine_factor=3e-5,
                             method="gcr")[0]
    if c["transpose"]:
        return state["H"].action_transpose_device(state["x"], precision=state["precision"])
    return state["H"].action_device(state["x"], precision=state["precision"])


# ---------------------------------------------------------------------------
# work

@functools.lru_cache(maxsize=64)
def _entries(dim, n, m, points, interp, deg, eta, kind):
    """Kernel entries of one action, near and far, counted by the host planner
    on one cloud of these sizes."""
    P, T = _points({"dim": dim, "n": n, "m": m, "points": points, "kind": kind}, 0)
    H = fmca_amd.H2kernelActor(fmca_amd.CovarianceKernel("MATERN32", 0.5),
                               P if T is None else T, P, deg, eta, interp, planner="host")
    info = H.info()
    return info["near_entries"] + info["far_entries"]


# products of one solve: GCR to 1e-8 at these ridges takes about 56 iterations
_SOLVE_PRODUCTS = 56


def work(case):
    e = _entries(case["dim"], case["n"], case["m"], case["points"], case["interp"], case["deg"],
                 case["eta"], case["kind"])
    r, d = case["nrhs"], case["dim"]
    rows = case["m"] or case["n"]
    pts = 8 * d * (case["n"] + case["m"])
    vecs = 8 * r * (case["n"] + rows)
    entry = 3 * d + 4  # squared distance, root, exponential, polynomial
    if case["kind"] == "assembled":
        size = 8 if case["precision"] == "FP64" else 4
        return {"bytes": size * e + vecs, "flops": 2 * r * e}
    if case["kind"] == "solve":
        return {"bytes": pts + vecs, "flops": _SOLVE_PRODUCTS * (2 * r + entry) * e}
    if case["kind"] == "step":
        # forward; backward: K^T G, the weights G_p . alpha_j of the entries
        # (for the lengthscale and the points) and their kernel derivatives
        flops = (2 * r + entry) * e + (4 * r + 2 * entry) * e
        return {"bytes": 2 * (pts + vecs), "flops": flops}
    return {"bytes": pts + vecs, "flops": (2 * r + entry) * e}


def tolerance(case):
    """Relative 2-norm distances, about four times the largest measured over
    these ranges: FP64 calls against the same columns in other groups (other
    kernels, other order of the sums) and against the dense sums, FP32 forms
    against FP64, solutions of other methods."""
    if case["kind"] == "solve":
        return {"rel": 2e-8}  # residuals of 1e-8; measured up to 7e-9
    if case["kind"] == "step":
        if case["precision"] == "FP64":
            return {"rel": 4e-13}  # the lengthscale's sum cancels: 1e-13
        if "p" in case["wrt"]:
            # FP32 differences of close points; phi(r) grows as 1 / r for a
            # kernel with a cusp at 0 (measured 2e-3)
            return {"rel": 8e-3 if case["ktype"] == "EXPONENTIAL" else 1e-4}
        return {"rel": 6e-5}  # the lengthscale's sum again: 1.5e-5
    if case["precision"] == "FP64":
        return {"rel": 3e-14}  # 6e-15
    return {"rel": 2.4e-5}  # FP32 4e-6, FP32_BF16 6e-6


# ---------------------------------------------------------------------------
# the dense matrix in 64 bits

def _profile(ktype, r2, l):
    """(k, k'(r) / r) of the squared distances; k'(r) / r is 0 at r = 0 where
    it is singular."""
    if ktype == "GAUSSIAN":
        k = torch.exp(r2 * (-0.5 / (l * l)))
        return k, k * (-1.0 / (l * l))
    if ktype == "INVMULTIQUADRIC":
        return 1.0 / torch.sqrt(r2 / (l * l) + 1.0), None
    r = torch.sqrt(r2)
    if ktype == "EXPONENTIAL":
        k = torch.exp(r / (-l))
        return k, torch.where(r > 0, k / (r * (-l)), torch.zeros_like(r))
    s = {"MATERN32": 3.0, "MATERN52": 5.0, "MATERN72": 7.0, "MATERN92": 9.0}[ktype] ** 0.5 / l
    x = r * s
    e = torch.exp(-x)
    if ktype == "MATERN32":
        return (1 + x) * e, -s * s * e
    if ktype == "MATERN52":
        return (1 + x + x * x / 3) * e, -s * s / 3 * (1 + x) * e
    if ktype == "MATERN72":
        return (1 + x + 2 * x * x / 5 + x * x * x / 15) * e, None
    return (1 + x + 3 * x * x / 7 + 2 * x ** 3 / 21 + x ** 4 / 105) * e, None


def _dense(case, T, P, x):
    """K(T, P) x."""
    out = torch.empty((T.shape[1], x.shape[1]), dtype=torch.float64, device="cuda")
    step = max(1, 64_000_000 // P.shape[1])
    for i in range(0, T.shape[1], step):
        r2 = sum((T[d, i:i + step, None] - P[d]).square_() for d in range(T.shape[0]))
        out[i:i + step] = _profile(case["ktype"], r2, case["l"])[0] @ x
    return out


def _dense_step(case, T, P, a, G):
    """K a, K^T G, <G, dK/dl a> and the gradients in the sources and targets."""
    l = case["l"]
    y = torch.empty((T.shape[1], a.shape[1]), dtype=torch.float64, device="cuda")
    da = torch.zeros_like(a)
    dl = torch.zeros((), dtype=torch.float64, device="cuda")
    dP, dT = torch.zeros_like(P), torch.zeros_like(T)
    step = max(1, 32_000_000 // P.shape[1])
    for i in range(0, T.shape[1], step):
        diff = [T[d, i:i + step, None] - P[d] for d in range(T.shape[0])]
        r2 = sum(x * x for x in diff)
        k, phi = _profile(case["ktype"], r2, l)
        g = G[i:i + step]
        y[i:i + step] = k @ a
        da += (g.t().contiguous() @ k).t()
        if case["ktype"] == "EXPONENTIAL":
            dk = k * torch.sqrt(r2) / (l * l)
        else:
            dk = r2 * phi / (-l)
        w = g @ a.t().contiguous()
        dl += (w * dk).sum()
        w *= phi
        for d, x in enumerate(diff):
            wx = w * x
            dT[d, i:i + step] = wx.sum(1)
            dP[d] -= wx.sum(0)
    return y, da, dl, dP, dT


def exact(case, seed):
    rows = case["m"] or case["n"]
    kind = case["kind"]
    if kind == "solve" or case["n"] * rows > (4.1e10 if kind == "step" else 1.0e11):
        return None
    P, T = _points(case, seed)
    Pd = torch.from_numpy(np.ascontiguousarray(P)).cuda()
    Td = Pd if T is None else torch.from_numpy(np.ascontiguousarray(T)).cuda()
    if kind in ("oneshot", "evaluate"):
        x = torch.from_numpy(np.ascontiguousarray(_host_rhs(case, seed))).cuda()
        return _dense(case, Td, Pd, x).cpu().numpy()
    if kind == "step":
        a = _rhs(case, seed).contiguous()
        G = _normal(rows, case["nrhs"], seed + 2).contiguous()
        y, da, dl, dP, dT = _dense_step(case, Td, Pd, a, G)
        out = [y, da, dl]
        if "p" in case["wrt"]:
            out += [dP + dT] if T is None else [dP, dT]
        return out
    x = _rhs(case, seed).contiguous()
    return _dense(case, Pd, Td, x) if case["transpose"] else _dense(case, Td, Pd, x)
