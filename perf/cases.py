"""The work that users of this framework give it, as cases to time.

A case is a dict of plain values; prepare(case, seed) builds what a program
holds before the call (handles, device buffers), run(state) makes one pass
through the package's public entry points, work(case) says what a pass cannot
do without, and exact(case, seed) computes the same outputs in 64 bits with
plain torch and numpy (the discontinuous Galerkin operator of the Euler
equations on boxes, warped boxes and quadrilaterals, and the closure network).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dg-mpi_amd"))

GAMMA = 1.4
NF, NH, NO = 70, 128, 40          # the closure network's features, hidden width, outputs
CFL = {1: 0.1, 2: 0.1, 3: 0.06, 4: 0.03, 5: 0.02}   # stable on the flows below


def listed():
    return [
        # one RK4 step of a small box: a program that steps and looks at the state each time
        {"name": "step_8c_p2", "kind": "step", "nx": 8, "ny": 8, "nz": 8, "order": 2, "basis": "LegendreHex",
         "flux": "Roe", "ic": "vortex", "precision": "FP64", "steps": 1},
        # a small ragged box marched many steps in one call, nodal basis
        {"name": "march_9x11x7_p3", "kind": "step", "nx": 9, "ny": 11, "nz": 7, "order": 3, "basis": "LagrangeHex",
         "flux": "HLLC", "ic": "vortex", "precision": "FP64", "steps": 20},
        # the headline configuration, in FP64 and in the FP32 form
        {"name": "step_64c_p3", "kind": "step", "nx": 64, "ny": 64, "nz": 64, "order": 3, "basis": "LegendreHex",
         "flux": "Roe", "ic": "vortex", "precision": "FP64", "steps": 1},
        {"name": "step_64c_p3_fp32", "kind": "step", "nx": 64, "ny": 64, "nz": 64, "order": 3, "basis": "LegendreHex",
         "flux": "Roe", "ic": "vortex", "precision": "FP32", "steps": 1},
        # the low-order run: a density bump carried over 64^3 elements
        {"name": "step_64c_p1", "kind": "step", "nx": 64, "ny": 64, "nz": 64, "order": 1, "basis": "LegendreHex",
         "flux": "LaxFriedrichs", "ic": "bump", "precision": "FP64", "steps": 1},
        # the large high-order run: Taylor-Green at p = 4, 32.8 M DOF x 5
        {"name": "step_64c_p4", "kind": "step", "nx": 64, "ny": 64, "nz": 64, "order": 4, "basis": "LegendreHex",
         "flux": "Roe", "ic": "tgv", "precision": "FP64", "steps": 1},
        # a program with a stepper of its own: residual and inverse mass on its buffers, odd sizes, nodal basis
        {"name": "residual_45x37x51_p2", "kind": "residual", "nx": 45, "ny": 37, "nz": 51, "order": 2,
         "basis": "LagrangeHex", "flux": "HLLC", "ic": "vortex", "precision": "FP64"},
        # non-affine (trilinear) elements
        {"name": "warped_24x20x22_p3", "kind": "warped", "nx": 24, "ny": 20, "nz": 22, "order": 3,
         "basis": "LegendreHex", "flux": "LaxFriedrichs", "ic": "vortex", "steps": 1},
        # two space dimensions
        {"name": "quads_512_p3", "kind": "quads", "nx": 512, "ny": 512, "order": 3, "basis": "LegendreQuad",
         "flux": "Roe", "ic": "vortex2d", "steps": 1},
        # many independent uneven cases advanced together
        {"name": "batch_32", "kind": "batch", "cases": 32, "nmin": 8, "nmax": 20, "flux": "Roe",
         "basis": "LegendreHex", "precision": "FP64", "steps": 2},
        # the closure network: mini-batches of its training, and the corrected p = 1 step
        {"name": "closure_train_4096", "kind": "train", "batch": 4096, "batches": 8},
        {"name": "closure_step_32c", "kind": "closure", "n": 32, "steps": 1},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, dof_lo, dof_hi, order, dim=3):
    """Ragged edge lengths of a box with about so many degrees of freedom."""
    elems = max(8.0, _log_int(rng, dof_lo, dof_hi) / float((order + 1) ** dim))
    edge = elems ** (1.0 / dim)
    return [max(2, int(round(edge * rng.uniform(0.8, 1.25)))) for _ in range(dim)]


def draw(rng):
    kind = rng.choice(["step"] * 6 + ["residual", "warped", "quads", "batch", "train", "closure"])
    flux = rng.choice(["Roe", "Roe", "HLLC", "LaxFriedrichs"])
    basis = rng.choice(["LegendreHex", "LegendreHex", "LagrangeHex"])
    if kind in ("step", "residual"):
        order = rng.randint(1, 5)
        nx, ny, nz = _box(rng, 4e3, 1.2e7, order)
        prec = rng.choice(["FP64", "FP64", "FP64", "FP32", "FP32", "BF16"])
        c = {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "order": order, "basis": basis, "flux": flux,
             "ic": rng.choice(["vortex", "bump", "tgv"]), "precision": prec}
        if kind == "step":
            c["steps"] = rng.randint(1, 8) if nx * ny * nz * (order + 1) ** 3 < 3e5 else 1
        return c
    if kind == "warped":
        order = rng.randint(1, 4)
        nx, ny, nz = _box(rng, 4e3, 1e6, order)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "order": order, "basis": basis, "flux": flux,
                "ic": "vortex", "steps": 1}
    if kind == "quads":
        order = rng.randint(1, 5)
        nx, ny = _box(rng, 4e3, 6e6, order, 2)
        return {"kind": kind, "nx": nx, "ny": ny, "order": order, "basis": basis.replace("Hex", "Quad"),
                "flux": flux, "ic": "vortex2d", "steps": 1}
    if kind == "batch":
        return {"kind": kind, "cases": rng.randint(6, 40), "nmin": rng.randint(5, 9), "nmax": rng.randint(12, 20),
                "flux": flux, "basis": basis, "precision": rng.choice(["FP64", "FP64", "FP32"]), "steps": 2}
    if kind == "train":
        return {"kind": kind, "batch": _log_int(rng, 500, 6000), "batches": rng.randint(2, 8)}
    return {"kind": kind, "n": rng.randint(8, 32), "steps": rng.randint(1, 3)}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
# initial conditions of the package by the name used here
IC_NAMES = {"vortex": "ExtrudedIsentropicVortex", "bump": "GaussianBump", "tgv": "TaylorGreen",
            "vortex2d": "IsentropicVortex", "mix": "VortexPulseMix"}


def _ic_data(ic, rng):
    """Initial-condition data of a seed: centres, strengths and directions vary."""
    if ic == "vortex":
        u = float(rng.uniform(0.2, 0.8)) * math.sqrt(GAMMA / 2.0)
        return [1.0, u, u, 1.0, float(rng.uniform(1.0, 5.0))] + [float(v) for v in rng.uniform(-2.0, 2.0, 2)]
    if ic == "vortex2d":
        u = float(rng.uniform(0.2, 0.8)) * math.sqrt(GAMMA / 2.0)
        return [1.0, u, u, 1.0, float(rng.uniform(1.0, 5.0))]
    if ic == "bump":
        d = rng.normal(size=3)
        d *= 1.0 / np.linalg.norm(d)
        return [0.2, 1.5] + [float(v) for v in d] + [1.0 / GAMMA] + [float(v) for v in rng.uniform(-2.0, 2.0, 3)]
    if ic == "tgv":
        return [float(rng.uniform(0.08, 0.12))]
    nv = int(rng.integers(1, 5))
    d = [float(rng.uniform(-0.5, 0.5)), float(rng.uniform(-0.5, 0.5))]
    for k in range(4):
        c = rng.uniform(-5.0, 5.0, 2)
        d += [float(c[0]), float(c[1]), float(rng.uniform(1.0, 5.0)) if k < nv else 0.0]
    return d + [float(rng.uniform(0.01, 0.05))] + [float(v) for v in rng.uniform(-5.0, 5.0, 3)] + [1.0]


def _box_case(c, seed):
    """What the text of one box case and its 64-bit counterpart are made from."""
    rng = np.random.default_rng(seed)
    dim = 2 if c["kind"] == "quads" else 3
    ne = [c["nx"], c["ny"]] + ([c["nz"]] if dim == 3 else [])
    lo, hi = (0.0, 2.0 * math.pi) if c["ic"] == "tgv" else (-5.0, 5.0)
    data = _ic_data(c["ic"], rng)
    speed = 1.0 + 1.0 / data[0] if c["ic"] == "tgv" else 3.0   # about the largest |u| + c
    return {"dim": dim, "ne": ne, "lo": lo, "hi": hi, "order": c["order"], "basis": c["basis"], "flux": c["flux"],
            "ic": c["ic"], "data": data, "dt": CFL[c["order"]] * (hi - lo) / max(ne) / speed,
            "warp": 0.1 if c["kind"] == "warped" else 0.0, "precision": c.get("precision", "FP64")}


def _solver(b):
    import dg_amd
    prec = None if b["precision"] == "FP64" else b["precision"]
    s = dg_amd.Solver(dg_amd.case_toml(order=b["order"], basis=b["basis"], flux=b["flux"], nelem=b["ne"],
                                       lower=[b["lo"]] * b["dim"], upper=[b["hi"]] * b["dim"], timestep=b["dt"],
                                       ic=IC_NAMES[b["ic"]], ic_data=b["data"], warp=b["warp"],
                                       normals="exact" if b["warp"] else "reference", precision=prec))
    s.init_state_from_fcn()
    return s


class _StateArray:
    """The state of a handle where it lies, for torch.as_tensor; keeps the handle alive."""

    def __init__(self, solver):
        self.solver = solver
        self.__cuda_array_interface__ = {"shape": tuple(solver.shape), "typestr": "<f8", "version": 3,
                                         "strides": None, "data": (solver.state_device_ptr(), False)}


def _state(solver):
    return torch.as_tensor(_StateArray(solver), device="cuda")


def _batch_members(c, seed):
    """The uneven cases of a batch: sizes from the case alone, flows from the seed."""
    sizes = np.random.default_rng(c["cases"] * 1000 + c["nmax"])
    out = []
    for k in range(c["cases"]):
        n, p = int(sizes.integers(c["nmin"], c["nmax"] + 1)), int(sizes.integers(1, 5))
        out.append({"kind": "step", "nx": n, "ny": n, "nz": n, "order": p, "basis": c["basis"], "flux": c["flux"],
                    "ic": "vortex", "precision": c["precision"], "steps": c["steps"]})
    return [_box_case(m, seed * 1000 + k) for k, m in enumerate(out)]


class _Batch:
    """A batch and its cases, given back in order."""

    def __init__(self, boxes):
        import dg_amd
        self.solvers = [_solver(b) for b in boxes]
        self.batch = dg_amd.Batch(self.solvers)
        self.out = [_state(s) for s in self.solvers]

    def __del__(self):
        if getattr(self, "batch", None) is not None:
            self.batch.close()


def _network(rng):
    """Parameters of a network in training: He-normal hidden layers, a small output layer, small biases."""
    w1, w2 = rng.normal(size=(NF, NH)) * math.sqrt(2.0 / NF), rng.normal(size=(NH, NH)) * math.sqrt(2.0 / NH)
    w3 = rng.normal(size=(NH, NO)) * math.sqrt(1.0 / NH)
    parts = [w1, 0.1 * rng.normal(size=NH), w2, 0.1 * rng.normal(size=NH), w3, 0.1 * rng.normal(size=NO)]
    return np.concatenate([v.ravel() for v in parts]).astype(np.float32)


def _train_inputs(c, seed):
    rng = np.random.default_rng(seed)
    rows = c["batch"] * c["batches"]
    mean, std = rng.normal(size=NF).astype(np.float32), np.exp(rng.normal(size=NF)).astype(np.float32)
    ys = np.exp(rng.normal(size=NO) - 3.0).astype(np.float32)
    z = rng.normal(size=(rows, NF)).astype(np.float32)
    x = mean + std * z
    y = ys * np.tanh(z[:, :NO] + 0.5 * z[:, NF - NO:]).astype(np.float32)
    return {"p": _network(rng), "mean": mean, "scale": (1.0 / std).astype(np.float32), "ys": ys,
            "x": x.astype(np.float32), "y": y.astype(np.float32), "idx": rng.permutation(rows).astype(np.int32)}


LR = 1e-3


def _closure_inputs(c, seed):
    rng = np.random.default_rng(seed)
    b = {"dim": 3, "ne": [c["n"]] * 3, "lo": -5.0, "hi": 5.0, "order": 1, "basis": "LegendreHex", "flux": "Roe",
         "ic": "mix", "data": _ic_data("mix", rng), "dt": 0.1 * 10.0 / c["n"] / 3.0, "warp": 0.0, "precision": "FP64"}
    mean = np.zeros(NF, np.float32)
    mean[[0, 4]] = 1.0, 2.5
    return b, {"p": _network(rng), "mean": mean, "scale": np.full(NF, 5.0, np.float32),
               "ys": np.full(NO, 1e-3, np.float32)}


def _mlp(d):
    from dg_amd import closure
    m = closure.MLP(0)
    m.set_params(d["p"])
    m.set_scaling(d["mean"], d["scale"], d["ys"])
    return m


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("step", "warped", "quads"):
        s = _solver(_box_case(case, seed))
        return {"case": case, "solver": s, "out": _state(s)}
    if kind == "residual":
        b = _box_case(case, seed)
        s = _solver(b)
        u = _state(s).clone()
        torch.cuda.synchronize()
        return {"case": case, "solver": s, "dt": b["dt"], "u": u, "r": torch.empty_like(u), "du": torch.empty_like(u)}
    if kind == "batch":
        return {"case": case, "batch": _Batch(_batch_members(case, seed))}
    from dg_amd import hip
    if kind == "train":
        d = _train_inputs(case, seed)
        return {"case": case, "mlp": _mlp(d), "x": hip.Buffer.from_array(d["x"], np.float32),
                "y": hip.Buffer.from_array(d["y"], np.float32), "idx": hip.Buffer.from_array(d["idx"], np.int32)}
    b, d = _closure_inputs(case, seed)
    s = _solver(b)
    return {"case": case, "solver": s, "mlp": _mlp(d), "out": _state(s)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("step", "warped", "quads"):
        state["solver"].take_time_step(0.0, case["steps"])
        return state["out"]
    if kind == "residual":
        s = state["solver"]
        s.get_residual(state["u"].data_ptr(), state["r"].data_ptr())
        s.mult_inv_mass_matrix(state["dt"], state["r"].data_ptr(), state["du"].data_ptr())
        return {"r": state["r"], "du": state["du"]}
    if kind == "batch":
        state["batch"].batch.step(case["steps"])
        return state["batch"].out
    from dg_amd import closure
    if kind == "train":
        m = state["mlp"]
        loss = m.train(state["x"], state["y"], case["batch"] * case["batches"], state["idx"], case["batch"], LR)
        return {"loss": float(loss), "params": m.params()}
    closure.step(state["solver"], state["mlp"], 1e30, case["steps"])
    return state["out"]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _stage_flops(p, dim):
    """Sum-factorised residual of one element: interpolation and weak gradient lines, point and face fluxes."""
    n, m, v = p + 1, p + 2, dim + 2
    if dim == 3:
        lines = n ** 3 * m + n ** 2 * m ** 2 + n * m ** 3
        return 2 * v * 4 * lines + 2 * 12 * v * (n ** 3 + n * n * m + n * m * m) + 60 * m ** 3 + 300 * m * m
    lines = n * n * m + n * m * m
    return 2 * v * 3 * lines + 2 * 8 * v * (n * n + n * n) + 40 * m * m + 250 * n


def _step_work(ne, p, dim, steps, precision="FP64", dense=False):
    """RK4 with the registers of its textbook form: 17 passes over the state in four stages (U, stage states and the
    accumulator), and in the reduced forms the 32-bit rounding error read and written once a step."""
    elems = float(np.prod(ne))
    values = elems * (p + 1) ** dim * (dim + 2)
    bytes_ = 17.0 * 8.0 * values + (0.0 if precision == "FP64" else 8.0 * values)
    flops = 4.0 * elems * _stage_flops(p, dim)
    if dense:      # nodes, face records and one dense inverse mass matrix per element and stage
        nb = (p + 1) ** dim
        bytes_ += 4.0 * elems * (8.0 * nb * nb + 8.0 * 24 + 48)
        flops += 4.0 * elems * (2.0 * nb * nb * 5 + 150.0 * ((p + 2) ** 3 + 6 * (p + 2) ** 2))
    return {"bytes": bytes_ * steps, "flops": flops * steps}


def work(case):
    kind = case["kind"]
    if kind in ("step", "warped"):
        return _step_work([case["nx"], case["ny"], case["nz"]], case["order"], 3, case["steps"],
                          case.get("precision", "FP64"), kind == "warped")
    if kind == "quads":
        return _step_work([case["nx"], case["ny"]], case["order"], 2, case["steps"])
    if kind == "residual":     # U read and R written, then R read and dU written
        elems = float(case["nx"] * case["ny"] * case["nz"])
        values = elems * (case["order"] + 1) ** 3 * 5
        return {"bytes": 4 * 8 * values, "flops": elems * _stage_flops(case["order"], 3) + 2 * values}
    if kind == "batch":
        each = [_step_work(b["ne"], b["order"], 3, case["steps"], case["precision"]) for b in _batch_members(case, 1)]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    weights = NF * NH + NH * NH + NH * NO
    if kind == "train":        # each row once, parameters and both moments read and written per mini-batch
        rows = case["batch"] * case["batches"]
        return {"bytes": 4.0 * rows * (NF + NO + 1) + 24.0 * weights * case["batches"], "flops": 6.0 * rows * weights}
    elems = float(case["n"] ** 3)
    w = _step_work([case["n"]] * 3, 1, 3, case["steps"])
    return {"bytes": w["bytes"], "flops": w["flops"] + 4 * case["steps"] * 2.0 * elems * weights}


# ---------------------------------------------------------------------------
# The same in 64 bits with plain torch
# ---------------------------------------------------------------------------
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=_dev())


def _basis(name, p, x):
    """Values and derivatives [len(x)][p + 1] of the 1D basis: Legendre polynomials or Lagrange on equidistant nodes."""
    x = np.asarray(x, float)
    if name.startswith("Legendre"):
        polys = [np.polynomial.legendre.Legendre.basis(i) for i in range(p + 1)]
    else:
        nodes = np.linspace(-1.0, 1.0, p + 1)
        polys = []
        for i in range(p + 1):
            q = np.polynomial.Polynomial.fromroots(np.delete(nodes, i))
            polys.append(q / q(nodes[i]))
    return np.stack([q(x) for q in polys], 1), np.stack([q.deriv()(x) for q in polys], 1)


def _along(mat, u, axis):
    """sum_i mat[a][i] u[.. i ..] along an axis."""
    return torch.movedim(torch.tensordot(u, mat, dims=([axis], [1])), -1, axis)


def _pressure(u):
    mom = u[..., 1:-1]
    return (GAMMA - 1.0) * (u[..., -1] - 0.5 * (mom * mom).sum(-1) / u[..., 0])


def _flux_n(u, n):
    """Euler flux along the unit normal n [.., dim]."""
    p = _pressure(u)
    un = (u[..., 1:-1] * n).sum(-1) / u[..., 0]
    return torch.cat([(u[..., 0] * un)[..., None], u[..., 1:-1] * un[..., None] + p[..., None] * n,
                      ((u[..., -1] + p) * un)[..., None]], -1)


def _numerical(flux, ul, ur, n):
    """Numerical flux along the unit normal n: local Lax-Friedrichs, HLLC with pressure-based speeds, or Roe with an
    entropy fix on the acoustic waves."""
    rl, rr = ul[..., 0], ur[..., 0]
    pl, pr = _pressure(ul), _pressure(ur)
    vl, vr = ul[..., 1:-1] / rl[..., None], ur[..., 1:-1] / rr[..., None]
    cl, cr = torch.sqrt(GAMMA * pl / rl), torch.sqrt(GAMMA * pr / rr)
    nl, nr = (vl * n).sum(-1), (vr * n).sum(-1)
    fl, fr = _flux_n(ul, n), _flux_n(ur, n)
    if flux == "LaxFriedrichs":
        a = torch.maximum((vl * vl).sum(-1).sqrt() + cl, (vr * vr).sum(-1).sqrt() + cr)
        return 0.5 * (fl + fr) - 0.5 * a[..., None] * (ur - ul)
    if flux == "HLLC":
        ps = torch.clamp(0.5 * (pl + pr - (nr - nl) * 0.25 * (rl + rr) * (cl + cr)), min=0.0)
        g = (GAMMA + 1.0) / (2.0 * GAMMA)
        sl = nl - cl * torch.sqrt(1.0 + g * torch.clamp(ps / pl - 1.0, min=0.0))
        sr = nr + cr * torch.sqrt(1.0 + g * torch.clamp(ps / pr - 1.0, min=0.0))
        sm = (pr - pl + rl * nl * (sl - nl) - rr * nr * (sr - nr)) / (rl * (sl - nl) - rr * (sr - nr))

        def star(u, r, v, p, s, f):
            fac = r * (s - v) / (s - sm)
            us = torch.cat([torch.ones_like(fac)[..., None],
                            u[..., 1:-1] / r[..., None] + (sm - v)[..., None] * n,
                            (u[..., -1] / r + (sm - v) * (sm + p / (r * (s - v))))[..., None]], -1)
            return f + s[..., None] * (fac[..., None] * us - u)

        left = torch.where((sl >= 0)[..., None], fl, star(ul, rl, nl, pl, sl, fl))
        right = torch.where((sr <= 0)[..., None], fr, star(ur, rr, nr, pr, sr, fr))
        return torch.where(((sl >= 0) | ((sr > 0) & (sm >= 0)))[..., None], left, right)
    hl, hr = (ul[..., -1] + pl) / rl, (ur[..., -1] + pr) / rr
    wl = rl.sqrt() / (rl.sqrt() + rr.sqrt())
    v = wl[..., None] * vl + (1.0 - wl)[..., None] * vr
    h = wl * hl + (1.0 - wl) * hr
    q2 = (v * v).sum(-1)
    c = torch.sqrt((GAMMA - 1.0) * (h - 0.5 * q2))
    vn, r = (v * n).sum(-1), torch.sqrt(rl * rr)
    dr, dp, dn = rr - rl, pr - pl, nr - nl

    def fixed(lam, lam_l, lam_r):
        d = torch.clamp(torch.maximum(lam - lam_l, lam_r - lam), min=0.0)
        return torch.where(lam.abs() < d, 0.5 * (lam * lam + d * d) / torch.where(d > 0, d, torch.ones_like(d)),
                           lam.abs())

    w1 = fixed(vn - c, nl - cl, nr - cr) * (dp - r * c * dn) / (2.0 * c * c)
    w5 = fixed(vn + c, nl + cl, nr + cr) * (dp + r * c * dn) / (2.0 * c * c)
    w2 = vn.abs() * (dr - dp / (c * c))
    dv = (vr - vl) - dn[..., None] * n
    ws = (vn.abs() * r)[..., None]
    diss = torch.cat([(w1 + w2 + w5)[..., None],
                      w1[..., None] * (v - c[..., None] * n) + w5[..., None] * (v + c[..., None] * n) +
                      w2[..., None] * v + ws * dv,
                      (w1 * (h - vn * c) + w5 * (h + vn * c) + 0.5 * w2 * q2 + ws[..., 0] * (v * dv).sum(-1))[..., None]],
                     -1)
    return 0.5 * (fl + fr) - 0.5 * diss


def _primitive(rho, vel, p):
    mom = rho[..., None] * vel
    e = p / (GAMMA - 1.0) + 0.5 * (mom * vel).sum(-1)
    return torch.cat([rho[..., None], mom, e[..., None]], -1)


def _initial(b, x):
    """The initial condition at points x [.., dim]."""
    d, ic = b["data"], b["ic"]
    length = b["hi"] - b["lo"]

    def wrap(y):
        return y - length * torch.round(y / length)

    one = torch.ones_like(x[..., 0])
    if ic in ("vortex", "vortex2d"):
        xr, yr = x[..., 0], x[..., 1]
        if ic == "vortex":
            xr, yr = wrap(xr - d[5]), wrap(yr - d[6])
        e = torch.exp(0.5 * (1.0 - xr * xr - yr * yr))
        a = d[4] / (2.0 * math.pi) * e
        temp = d[3] / d[0] - (GAMMA - 1.0) * d[4] ** 2 / (8.0 * GAMMA * math.pi ** 2) * e * e
        rho = (temp / (d[3] / d[0] ** GAMMA)) ** (1.0 / (GAMMA - 1.0))
        vel = [d[1] - a * yr, d[2] + a * xr] + ([0.0 * one] if b["dim"] == 3 else [])
        return _primitive(rho, torch.stack(vel, -1), rho * temp)
    if ic == "bump":
        r2 = sum(wrap(x[..., k] - d[6 + k]) ** 2 for k in range(3))
        return _primitive(1.0 + d[0] * torch.exp(-r2 / d[1] ** 2), torch.stack([v * one for v in d[2:5]], -1), d[5] * one)
    if ic == "tgv":
        s, c = torch.sin(x), torch.cos(x)
        vel = torch.stack([s[..., 0] * c[..., 1] * c[..., 2], -c[..., 0] * s[..., 1] * c[..., 2], 0.0 * one], -1)
        p = 1.0 / (GAMMA * d[0] ** 2) + (torch.cos(2 * x[..., 0]) + torch.cos(2 * x[..., 2])) * (
            torch.cos(2 * x[..., 1]) + 2.0) / 16.0
        return _primitive(one, vel, p)
    u, v, temp = d[0] * one, d[1] * one, one.clone()
    for k in range(4):
        xr, yr = wrap(x[..., 0] - d[2 + 3 * k]), wrap(x[..., 1] - d[3 + 3 * k])
        e = torch.exp(0.5 * (1.0 - xr * xr - yr * yr))
        a = d[4 + 3 * k] / (2.0 * math.pi) * e
        u, v = u - a * yr, v + a * xr
        temp = temp - (GAMMA - 1.0) * d[4 + 3 * k] ** 2 / (8.0 * GAMMA * math.pi ** 2) * e * e
    rho = temp ** (1.0 / (GAMMA - 1.0))
    pulse = d[14] * torch.exp(-sum(wrap(x[..., k] - d[15 + k]) ** 2 for k in range(3)) / d[18] ** 2)
    return _primitive(rho + pulse / GAMMA, torch.stack([u, v, 0.0 * one], -1), rho * temp + pulse)


class _BoxOperator:
    """The DG operator on a periodic box of affine elements; states [nz][ny][nx][k][j][i][variable]."""

    def __init__(self, b):
        self.b, self.dim = b, b["dim"]
        p, dim = b["order"], b["dim"]
        self.h = [(b["hi"] - b["lo"]) / n for n in b["ne"]]
        self.jac = float(np.prod([0.5 * v for v in self.h]))
        x, w = np.polynomial.legendre.leggauss(p + 2)
        val, der = _basis(b["basis"], p, x)
        self.B, self.Bw, self.Dw = _t(val), _t((val * w[:, None]).T), _t((der * w[:, None]).T)
        x, w = np.polynomial.legendre.leggauss(p + 2 if dim == 3 else p + 1)   # faces
        val, _ = _basis(b["basis"], p, x)
        self.Bf, self.Bfw = _t(val), _t((val * w[:, None]).T)
        self.ends = [_t(_basis(b["basis"], p, [e])[0]) for e in (-1.0, 1.0)]
        self.xq, self.wq = np.polynomial.legendre.leggauss(2 * p + 2)
        self.BQ = _basis(b["basis"], p, self.xq)[0]
        self.Minv = _t(np.linalg.inv(self.BQ.T @ (self.BQ * self.wq[:, None])))

    def elem_axis(self, d):
        return self.dim - 1 - d

    def mode_axis(self, d):
        return 2 * self.dim - 1 - d

    def inv_mass(self, r):
        for d in range(self.dim):
            r = _along(self.Minv, r, self.mode_axis(d))
        return r / self.jac

    def initial(self):
        dim, xs = self.dim, []
        for d in range(dim):
            n = self.b["ne"][d]
            shape = [1] * (2 * dim)
            shape[self.elem_axis(d)], shape[self.mode_axis(d)] = n, len(self.xq)
            pts = self.b["lo"] + (np.arange(n)[:, None] + 0.5 * (self.xq[None, :] + 1.0)) * self.h[d]
            xs.append(_t(pts).reshape(shape))
        u = _initial(self.b, torch.stack(torch.broadcast_tensors(*xs), -1))
        proj = _t((self.BQ * self.wq[:, None]).T)
        for d in range(dim):
            u = _along(proj, u, self.mode_axis(d))
        return self.inv_mass(u * self.jac)

    def residual(self, u):
        dim = self.dim
        uq = u
        for d in range(dim):
            uq = _along(self.B, uq, self.mode_axis(d))
        r = torch.zeros_like(u)
        for d in range(dim):
            n = torch.zeros(dim, dtype=torch.float64, device=u.device)
            n[d] = 1.0
            g = _flux_n(uq, n) * (2.0 / self.h[d] * self.jac)
            for k in range(dim):
                g = _along(self.Dw if k == d else self.Bw, g, self.mode_axis(k))
            r += g
            del g
            # the + face of every element, its neighbour across it the right one
            ul, ur = _along(self.ends[1], u, self.mode_axis(d)), _along(self.ends[0], u, self.mode_axis(d))
            for k in range(dim):
                if k != d:
                    ul, ur = _along(self.Bf, ul, self.mode_axis(k)), _along(self.Bf, ur, self.mode_axis(k))
            f = _numerical(self.b["flux"], ul, torch.roll(ur, -1, self.elem_axis(d)), n)
            f = f * float(np.prod([0.5 * self.h[k] for k in range(dim) if k != d]))
            for k in range(dim):
                if k != d:
                    f = _along(self.Bfw, f, self.mode_axis(k))
            r -= _along(self.ends[1].T.contiguous(), f, self.mode_axis(d))
            r += torch.roll(_along(self.ends[0].T.contiguous(), f, self.mode_axis(d)), 1, self.elem_axis(d))
        return r

    def flat(self, u):
        return u.reshape(int(np.prod(self.b["ne"])), -1, self.dim + 2)


class _WarpedOperator:
    """The same on the warped periodic box: trilinear elements, dense mass matrices, normals at the flux points;
    states [element][basis][variable]."""

    def __init__(self, b):
        self.b = b
        p, ne = b["order"], b["ne"]
        h = [(b["hi"] - b["lo"]) / n for n in ne]
        idx = np.meshgrid(*[np.arange(n + 1) for n in ne], indexing="ij")           # [i][j][k]
        turn = [2.0 * np.pi * (idx[d] % ne[d]) / ne[d] for d in range(3)]
        grid = np.stack([b["lo"] + idx[d] * h[d] + b["warp"] * h[d] * np.sin(turn[(d + 1) % 3]) *
                         np.sin(turn[(d + 2) % 3]) for d in range(3)], -1).transpose(2, 1, 0, 3)   # [k][j][i][xyz]
        nx, ny, nz = ne
        self.X = _t(np.stack([grid[c:c + nz, bb:bb + ny, a:a + nx].reshape(-1, 3)
                              for c in (0, 1) for bb in (0, 1) for a in (0, 1)], 1))    # node 4k + 2j + i
        x, w = np.polynomial.legendre.leggauss(p + 2)
        self.pts, self.w = self._tensor(x, x, x), _t(np.einsum("c,b,a->cba", w, w, w).ravel())
        self.val, self.grad = self._functions(x, x, x)
        q, wq = np.polynomial.legendre.leggauss(2 * p + 2)
        self.qval, _ = self._functions(q, q, q)
        qpts = self._tensor(q, q, q)
        self.qw, self.qx = _t(np.einsum("c,b,a->cba", wq, wq, wq).ravel()), self._map(qpts)
        self.qdet = (self._columns(qpts)[..., 0, :] * self._cofactors(qpts)[..., 0, :]).sum(-1)
        wd = self.qdet * self.qw
        mass = torch.stack([self.qval.T @ (v[:, None] * self.qval) for v in wd])
        self.Minv = _t(np.linalg.inv(mass.cpu().numpy()))
        self.cof = self._cofactors(self.pts)                                          # [e][q][d][xyz]
        self.faces = []
        for d in range(3):
            at = [x, x, x]
            at[d] = np.array([1.0])
            plus, (left, _) = self._tensor(*at), self._functions(*at)
            at[d] = np.array([-1.0])
            right, _ = self._functions(*at)
            wf = [w, w, w]
            wf[d] = np.array([1.0])
            e = np.arange(nx * ny * nz).reshape(nz, ny, nx)
            nbr = torch.as_tensor(np.roll(e, -1, 2 - d).ravel(), device=_dev())
            self.faces.append((left, right, _t(np.einsum("c,b,a->cba", wf[2], wf[1], wf[0]).ravel()),
                               self._cofactors(plus)[:, :, d, :], nbr))

    @staticmethod
    def _tensor(x, y, z):
        c, b, a = np.meshgrid(z, y, x, indexing="ij")
        return np.stack([a.ravel(), b.ravel(), c.ravel()], -1)

    def _functions(self, x, y, z):
        (vx, gx), (vy, gy), (vz, gz) = (_basis(self.b["basis"], self.b["order"], v) for v in (x, y, z))

        def prod(a, b, c):
            return _t(np.einsum("ck,bj,ai->cbakji", c, b, a).reshape(len(z) * len(y) * len(x), -1))
        return prod(vx, vy, vz), [prod(gx, vy, vz), prod(vx, gy, vz), prod(vx, vy, gz)]

    def _shapes(self, pts, d=None):
        """Trilinear shape functions (or their derivative along d) [point][node 4k + 2j + i]."""
        out = np.ones((len(pts), 8))
        for n in range(8):
            for k in range(3):
                s = 1.0 if (n >> k) & 1 else -1.0
                out[:, n] *= 0.5 * s if k == d else 0.5 * (1.0 + s * pts[:, k])
        return _t(out)

    def _map(self, pts):
        return torch.einsum("qn,enr->eqr", self._shapes(pts), self.X)

    def _columns(self, pts):
        return torch.stack([torch.einsum("qn,enr->eqr", self._shapes(pts, d), self.X) for d in range(3)], 2)

    def _cofactors(self, pts):
        a = self._columns(pts)
        return torch.stack([torch.linalg.cross(a[:, :, (d + 1) % 3], a[:, :, (d + 2) % 3], dim=-1) for d in range(3)], 2)

    def initial(self):
        f = _initial(self.b, self.qx) * (self.qdet * self.qw)[..., None]
        return self.inv_mass(torch.einsum("qb,eqs->ebs", self.qval, f))

    def inv_mass(self, r):
        return torch.matmul(self.Minv, r)

    def residual(self, u):
        uq = torch.einsum("qb,ebs->eqs", self.val, u)
        r = torch.zeros_like(u)
        for d in range(3):
            size = self.cof[:, :, d].norm(dim=-1, keepdim=True)
            g = _flux_n(uq, self.cof[:, :, d] / size) * size * self.w[:, None]
            r += torch.einsum("qb,eqs->ebs", self.grad[d], g)
            left, right, w, n, nbr = self.faces[d]
            size = n.norm(dim=-1, keepdim=True)
            f = _numerical(self.b["flux"], torch.einsum("qb,ebs->eqs", left, u),
                           torch.einsum("qb,ebs->eqs", right, u)[nbr], n / size) * size * w[:, None]
            r -= torch.einsum("qb,eqs->ebs", left, f)
            r.index_add_(0, nbr, torch.einsum("qb,eqs->ebs", right, f))
        return r

    def flat(self, u):
        return u


def _rk4(tendency, u, dt, steps):
    for _ in range(steps):
        k1 = tendency(u)
        k2 = tendency(u + 0.5 * dt * k1)
        k3 = tendency(u + 0.5 * dt * k2)
        k4 = tendency(u + dt * k3)
        u = u + dt / 6.0 * (k1 + 2.0 * k2 + 2.0 * k3 + k4)
    return u


def _bf16(v):
    return v.to(torch.float32).to(torch.bfloat16).to(torch.float64)


def _unpack(p):
    out, at = [], 0
    for shape in ((NF, NH), (NH,), (NH, NH), (NH,), (NH, NO), (NO,)):
        n = int(np.prod(shape))
        out.append(p[at:at + n].reshape(shape))
        at += n
    return out


def _net(p, x, mean, scale):
    """Normalised outputs of the network with its weights as they are used (rounded to bf16)."""
    w1, b1, w2, b2, w3, b3 = _unpack(p)
    h = torch.nn.functional.gelu((x - mean) * scale @ _bf16(w1) + b1)
    h = torch.nn.functional.gelu(h @ _bf16(w2) + b2)
    return h @ _bf16(w3) + b3


def _exact_train(case, seed):
    d = _train_inputs(case, seed)
    mean, scale, ys, x, y = (_t(d[k]) for k in ("mean", "scale", "ys", "x", "y"))
    p = _t(d["p"])
    m1, m2, total = torch.zeros_like(p), torch.zeros_like(p), 0.0
    idx = torch.as_tensor(d["idx"].astype(np.int64), device=p.device)
    for k in range(case["batches"]):
        rows = idx[k * case["batch"]:(k + 1) * case["batch"]]
        parts = _unpack(p)
        # the gradient is taken at the rounded weights and applied to the unrounded ones
        q = torch.cat([(_bf16(v) if i % 2 == 0 else v).reshape(-1) for i, v in enumerate(parts)]).requires_grad_(True)
        w1, b1, w2, b2, w3, b3 = _unpack(q)
        h = torch.nn.functional.gelu((x[rows] - mean) * scale @ w1 + b1)
        o = torch.nn.functional.gelu(h @ w2 + b2) @ w3 + b3
        loss = ((o - y[rows] / ys) ** 2).mean()
        g, = torch.autograd.grad(loss, q)
        total += float(loss.detach())
        m1, m2 = 0.9 * m1 + 0.1 * g, 0.999 * m2 + 0.001 * g * g
        p = p - LR * (m1 / (1.0 - 0.9 ** (k + 1))) / ((m2 / (1.0 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    return {"loss": total / case["batches"], "params": p}


def _exact_closure(case, seed):
    b, d = _closure_inputs(case, seed)
    op = _BoxOperator(b)
    p, mean, scale, ys = (_t(d[k]) for k in ("p", "mean", "scale", "ys"))

    def features(u):
        own = u.reshape(*u.shape[:3], 40)
        cols = [own]
        for ax in range(3):
            # face means of p = 1 Legendre states: the mean mode and the mode linear along the normal
            lin = [0, 0, 0]
            lin[2 - ax] = 1
            mean_mode, slope = u[:, :, :, 0, 0, 0], u[:, :, :, lin[0], lin[1], lin[2]]
            minus, plus = mean_mode - slope, mean_mode + slope
            cols += [torch.roll(plus, 1, 2 - ax) - minus, torch.roll(minus, -1, 2 - ax) - plus]
        return torch.cat(cols, -1)

    def tendency(u):
        c = _net(p, features(u).reshape(-1, NF), mean, scale) * ys
        return op.inv_mass(op.residual(u)) + c.reshape(u.shape)

    return op.flat(_rk4(tendency, op.initial(), b["dt"], case["steps"]))


def _exact_box(b, steps):
    op = _WarpedOperator(b) if b["warp"] else _BoxOperator(b)
    return op.flat(_rk4(lambda u: op.inv_mass(op.residual(u)), op.initial(), b["dt"], steps))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "warped", "quads"):
        return _exact_box(_box_case(case, seed), case["steps"])
    if kind == "residual":
        b = _box_case(case, seed)
        op = _BoxOperator(b)
        r = op.residual(op.initial())
        return {"r": op.flat(r), "du": op.flat(b["dt"] * op.inv_mass(r))}
    if kind == "batch":
        return [_exact_box(b, case["steps"]) for b in _batch_members(case, seed)]
    return _exact_train(case, seed) if kind == "train" else _exact_closure(case, seed)
