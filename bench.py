"""Benchmark of the DG residual + RK4 path on one MI355X.

Workload (the headline metric's configuration): 3D Euler, periodic cube
[-5,5]^3 with 64^3 hexahedra, LegendreHex p=3 (64 DOF/element, 16.8M DOF x
5 variables), Roe flux, classical RK4 at CFL 0.1 (dt from the initial
state), z-extruded isentropic vortex (rho=1, u=v=1, w=0, p=1, beta=5) --
synthetic, generated on the GPU.

A step is one RK4 step = 4 stages of two launches each (the faces, then the
elements; small boxes, BF16 and meshes: one launch).  W warm-up steps, then K
timed steps bracketed by stream synchronisation; HIP events are recorded on
the stream the stage kernels are launched on.

value = DOF-updates per second per RK stage = E (p+1)^3 / t_stage.

Accuracy: after the timed steps the run continues to 50 RK4 steps in all
(the configuration's count) and reports the L2 error against the exact
advected vortex.  Beside it, "fp32_form", "bf16x3_form", "bf16_form": the same run with
Numerics.precision = "FP32" (face and volume work of the stage kernel in
FP32, RK registers, M^-1 and the L2 reductions in FP64, compensated
update), "BF16x3" and "BF16" (the FP32 form with the x-y projection as a
bf16 matrix-core GEMM, hi/lo split or one term): rates, and L2 errors
against the FP64 run's; "gaussian_bump": the configuration's second
input (a density bump in uniform flow along a seeded direction), both
forms, 50 steps; "l2_err_vs_fp64_oracle": one RK4 step of both forms on a
32^3 box of the same case against the FP64 CPU oracle from the same state
(computed by the CPU-baseline leg, which times the oracle on that box).

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu]
Other workloads, one JSON line each: --batch 256 (batched uneven cases),
--closure 32 (learned closure: training and held-out evaluation),
--closure-timing 32 (cost of the corrected step against the plain one),
--tgv 96 (96^3 p=4 Taylor-Green to t=1, FP64 and FP32 forms, KE/mass drift).
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "dg-mpi_amd"))

METRIC = "DOF-updates/s per RK stage, Euler p=3 64^3 elems; L2 err vs FP64 oracle"
HBM_PEAK_GBS = 8000.0          # MI355X HBM3E, GB/s
FP64_PEAK_TFLOPS = 78.6        # MI355X FP64 vector
# algorithmic HBM bytes per DOF per stage: classical RK4 register passes
# (3 + 5 + 5 + 4) / 4 = 4.25 passes x 5 variables x 8 B
ALG_BYTES_PER_DOF = 4.25 * 5 * 8
P, NE = 3, 64
ORACLE_NE = 32                 # box of the oracle comparison and the CPU baseline sample
ACC_STEPS = 50                 # the configuration's step count: accuracy figures after 50 RK4 steps


def alg_flops_per_element(p):
    """Sum-factorised DG operator count per element per stage (affine)."""
    n, m, V = p + 1, p + 2, 5
    S = n ** 3 * m + n ** 2 * m ** 2 + n * m ** 3
    T = n ** 3 + n ** 2 * m + n * m ** 2
    return 2 * (4 * V * S + 12 * V * T) + 60 * m ** 3 + 300 * m ** 2 + 4 * V * n ** 3


def case_toml(ne, p=P, end=1.0, warp=0.0, dim=3, precision=None):
    import dg_amd
    if dim == 2:
        # the 2D path: ne x ne quadrilaterals, the reference's 2D vortex
        return dg_amd.case_toml(order=p, basis="LegendreQuad", flux="Roe", nelem=(ne, ne), lower=(-5., -5.),
                                upper=(5., 5.), stepper="RK4", cfl=0.1, end=end, ic="IsentropicVortex",
                                ic_data=(1.0, 1.0, 1.0, 1.0, 5.0))
    return dg_amd.case_toml(order=p, basis="LegendreHex", flux="Roe", nelem=(ne, ne, ne),
                            lower=(-5., -5., -5.), upper=(5., 5., 5.), stepper="RK4", cfl=0.1, end=end,
                            ic="ExtrudedIsentropicVortex", ic_data=(1.0, 1.0, 1.0, 1.0, 5.0), warp=warp,
                            precision=precision)


# elements from which an RK4 step runs in two passes (dg_kernels.hip,
# two_pass_min_elements), is split in halves up to (halves_team), and from
# which quadrilaterals go 16 to a wave (dg_kernels_2d.inc)
TWO_PASS_FROM = {"f64": (4608, 2560, 2816, 2816, 2816), "fp32": (7168, 5120, 5888, 14848, 8192)}
HALVES_TO = (2048, 1024, 768, 0, 0)
QUADS_FROM = (768, 2048, 3072, 2304, 2560)


def stage_kernels(order, E, dim, warp, precision):
    """(names of a stage's kernels, its number of launches)"""
    prec = (precision or "f64").lower()
    form = f"<{order},Roe" + ("" if prec == "f64" else ",fp32") + (f",{prec}" if prec.startswith("bf16") else "")
    if dim == 2:
        return ("stage2d_box_kernel" if E >= QUADS_FROM[order - 1] else "stage2d_kernel") + form + ">", 1
    if warp:
        return "stage_kernel" + form + ",mapped>", 1
    if not prec.startswith("bf16") and E >= TWO_PASS_FROM[prec][order - 1]:
        return f"face_flux_kernel{form}>+element_kernel{form.replace(',Roe', '')}>", 2
    if prec == "f64" and E <= HALVES_TO[order - 1]:
        return "stage_halves_kernel" + form + ">", 1
    return "stage_kernel" + form + ">", 1


def measured_traffic():
    """HBM bytes per stage from the committed rocprofv3 PMC summary,
    if present (profiles/stage_kernel_p3_64cube_traffic.json)."""
    f = os.path.join(ROOT, "profiles", "stage_kernel_p3_64cube_traffic.json")
    if os.path.exists(f):
        try:
            return json.load(open(f)).get("hbm_bytes_per_stage")
        except Exception:
            return None
    return None


def measured_copy_gbs():
    """Copy bandwidth this GPU reaches: dg-mpi_amd/bin/hbm_copy (a plain
    device-to-device copy kernel, 1 GiB read and 1 GiB written per launch),
    run as a child process; None where the tool is not built."""
    import subprocess
    exe = os.path.join(ROOT, "dg-mpi_amd", "bin", "hbm_copy")
    if not os.path.exists(exe):
        return None
    try:
        r = subprocess.run([exe, "1024", "20"], capture_output=True, text=True, timeout=120)
        return float(json.loads(r.stdout.strip().splitlines()[-1])["GBps"]) if r.returncode == 0 else None
    except (OSError, ValueError, KeyError, IndexError, subprocess.TimeoutExpired):
        return None


def cpu_model():
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return None


def legendre_l2(dU, ne, p, lo=-5.0, hi=5.0):
    """Volume-normalised L2 norm per variable of a LegendreHex coefficient
    difference dU[E][(p+1)^3][5] on the ne^3 box: for Legendre polynomials
    the integral of (sum c_b phi_b)^2 over an element is |J| sum_b c_b^2
    prod_d 2 / (2 i_d + 1), so the norm is exact for the polynomials."""
    import numpy as np
    n = p + 1
    i = np.arange(n)
    w1 = 2.0 / (2 * i + 1)
    wb = (w1[None, None, :] * w1[None, :, None] * w1[:, None, None]).ravel()     # b = i + n j + n^2 k
    h = (hi - lo) / ne
    jdet, vol = (h / 2) ** 3, (hi - lo) ** 3
    return np.sqrt(np.einsum("ebs,b->s", dU * dU, wb) * jdet / vol)


def cpu_baseline(gpu_step=None, budget_s=20.0):
    """The CPU oracle (reference algorithm restated, dense per-element
    GEMMs, OpenMP over elements) on a bounded sample of the workload: the
    same case on 32^3 elements, p=3, Roe, RK4, RK4 steps until ~budget_s.
    Its first step also checks the GPU: gpu_step = (U0, dt, {form: U1}) of
    one GPU RK4 step at 32^3 from U0; the difference of each form's U1 to the
    oracle's is returned as "L2 err vs FP64 oracle"."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import numpy as np
    import oracle as O
    ne = ORACLE_NE
    prm = O.make_params(order=P, basis="LegendreHex", flux="Roe", nelem=(ne, ne, ne), lo=(-5, -5, -5),
                        hi=(5, 5, 5), gamma=1.4, R=1.0, ic="ExtrudedIsentropicVortex", ic_data=(1, 1, 1, 1, 5))
    s = O.Solver(prm)
    check = None
    if gpu_step is not None:
        U0, dt, U1 = gpu_step
        s.set_state(U0)
    else:
        s.init_state()
        dt = 0.1 * (10.0 / ne) / s.max_wavespeed()
    steps, t0 = 0, time.perf_counter()
    while True:
        s.step("RK4", dt, 1)
        steps += 1
        if steps == 1 and gpu_step is not None:
            t_pause = time.perf_counter()
            ref = s.get_state()
            scale = float(np.max(np.abs(ref)))
            check = {"workload": f"one RK4 step of the same case at {ne}^3 (p=3 LegendreHex, Roe, dt of CFL 0.1) "
                                 "from the same initial state, GPU form vs the FP64 oracle",
                     "norm": "volume-normalised L2 norm of the state difference per variable (rho, rho u, rho v, "
                             "rho w, rho E), and max |difference| / max |oracle state|"}
            for form, U in U1.items():
                check[form] = {"l2": [float(x) for x in legendre_l2(U - ref, ne, P)],
                               "max_rel": float(np.max(np.abs(U - ref)) / scale)}
            del ref
            t0 += time.perf_counter() - t_pause       # the comparison is not CPU-baseline time
        el = time.perf_counter() - t0
        if el > budget_s or steps >= 50:
            break
    dof = ne ** 3 * (P + 1) ** 3
    threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
    base = {"value": dof * 4 * steps / el, "unit": "DOF-updates/s", "cores": threads, "kind": "port",
            "cpu_model": cpu_model(),
            "sample": f"oracle (dense reference formulation, OpenMP, {threads} threads) on {ne}^3 elements of the "
                      f"same case (p=3 LegendreHex, Roe, RK4), {steps} RK4 steps = {4 * steps} stages in {el:.1f} s"}
    return base, check


def io_bench(s, path):
    """Time dg_write_solution / dg_read_solution (data.h5, src/io/writer.cpp,
    src/solver/base.cpp:233-279) on the workload's state, device <-> file."""
    from dg_amd import h5
    import numpy as np
    nbytes = int(np.prod(s.shape)) * 8
    rec = {}
    for name, fn in (("write", lambda: s.write(path)), ("read", lambda: s.read_in_coefficients(path))):
        best = None
        for _ in range(3):
            t0 = time.perf_counter()
            fn()
            el = time.perf_counter() - t0
            best = el if best is None else min(best, el)
        rec[name] = {"s": best, "GB/s": nbytes / best / 1e9}
    print(json.dumps({"io": rec, "state_bytes": nbytes, "file_bytes": os.path.getsize(path),
                      "header": h5.read_header(path)}))


def batch_bench(args):
    """Batched uneven cases: 256 independent periodic vortex problems (seed
    args.seed) with n^3 elements, n uniform in 8..32 (8..args.batch_max_n), order p in {1..4},
    vortex centre (x, y) in [-2, 2]^2 (the vortex is z-extruded),
    vortex strength beta in [1, 5], free-stream Mach number in [0.2, 0.8]
    along (1, 1, 0) (rho = p = 1), Legendre, Roe, RK4 at CFL 0.1, 0.1, 0.06,
    0.04 for p = 1..4 (the dt = CFL h / max(|u| + c) rule is stable to these
    values over the whole Mach range; at Mach 0.2-0.5 CFL 0.1 is not at
    p = 3) -- advanced
    by dg_batch_step (one launch per order and RK stage, the order groups as
    concurrent branches of a captured HIP graph, team size and element
    bricks per group from the autotuner), against the same cases stepped
    one after the other with dg_step; then the same batch in the FP32 and
    BF16 forms against the FP64 one.  Per group: its rate run alone and its
    fraction of the HBM roofline.  Prints one JSON line."""
    import numpy as np
    import dg_amd
    from dg_amd import hip

    rng = np.random.default_rng(args.seed)
    n_cases = args.batch
    cases = []
    for _ in range(n_cases):
        n = int(rng.integers(8, args.batch_max_n + 1))
        p = int(rng.integers(1, 5))
        beta = float(rng.uniform(1.0, 5.0))
        mach = float(rng.uniform(0.2, 0.8))
        xc, yc = (float(v) for v in rng.uniform(-2.0, 2.0, 2))
        u = mach * np.sqrt(1.4) / np.sqrt(2.0)
        cases.append((n, p, beta, mach, (1.0, u, u, 1.0, beta, xc, yc)))

    def make(precision):
        out = []
        for n, p, beta, mach, data in cases:
            s = dg_amd.Solver(dg_amd.case_toml(order=p, basis="LegendreHex", flux="Roe", nelem=(n, n, n),
                                               cfl=(0.1, 0.1, 0.06, 0.04)[p - 1],
                                               ic="ExtrudedIsentropicVortex", ic_data=data, precision=precision))
            s.init_state_from_fcn()
            out.append(s)
        return out

    dof = sum(n ** 3 * (p + 1) ** 3 for n, p, *_ in cases)
    K, W = args.steps, max(args.warmup, 6)
    tunings, tiles = {}, {}

    def batch_time(solvers, key):
        # the warm-up call (6 steps at least) tunes team sizes and bricks
        with dg_amd.Batch(solvers) as b:
            b.step(W)
            hip.synchronize()
            t0 = time.perf_counter()
            b.step(K)
            tunings[key] = b.tuning()
            tiles[key] = b.tiles()
            return (time.perf_counter() - t0) / K

    def groups_of(key):
        # per group: its cases run alone at the chosen candidate (the tuning
        # timings), rate and fraction of the HBM roofline at 170 B per DOF
        # per stage (the FP64 register traffic of a stage)
        out = []
        for (o, team, a, b2), (cap, nc, ne, ms) in zip(tunings[key], tiles[key]):
            g_dof = sum(n ** 3 * (p + 1) ** 3 for n, p, *_ in cases if p == o)
            best = min(ms)
            out.append({"order": o, "cases": nc, "elements": ne, "dof": g_dof, "team": team,
                        "brick": f"{2 ** cap}^3 max", "ms_per_step_alone": best,
                        "ms_candidates": {f"team{c & 1}_brick{2 ** (3 - (c >> 1))}": m for c, m in enumerate(ms)},
                        "dof_updates_per_s": g_dof / (best / 4 * 1e-3),
                        "hbm_roofline_frac": ALG_BYTES_PER_DOF * g_dof / (best / 4 * 1e-3) / 1e9 / HBM_PEAK_GBS})
        return out

    s64 = make(None)
    t64 = batch_time(s64, "fp64")
    e64 = np.array([s.get_error()[0] for s in s64])
    s32 = make("FP32")
    t32 = batch_time(s32, "fp32")
    e32 = np.array([s.get_error()[0] for s in s32])
    d32 = np.array([float(np.max(np.abs(a.get_state() - b.get_state())) / np.max(np.abs(b.get_state())))
                    for a, b in zip(s32, s64)])
    for s in s32:
        s.close()
    sb = make("BF16")
    tb = batch_time(sb, "bf16")
    eb = np.array([s.get_error()[0] for s in sb])
    db = np.array([float(np.max(np.abs(a.get_state() - b.get_state())) / np.max(np.abs(b.get_state())))
                   for a, b in zip(sb, s64)])
    for s in sb:
        s.close()
    # the same FP64 cases one after the other (dg_step per case), same steps
    seq = make(None)
    for s in seq:
        s.take_time_step(0.0, W)
    hip.synchronize()
    t0 = time.perf_counter()
    for s in seq:
        s.take_time_step(0.0, K)
    hip.synchronize()
    t_seq = (time.perf_counter() - t0) / K
    same = max(float(np.max(np.abs(a.get_state() - b.get_state())) / np.max(np.abs(b.get_state())))
               for a, b in zip(s64, seq))
    for s in s64 + seq:
        s.close()
    ratio = e32 / e64
    ratio_b = eb / e64
    out = {
        "metric": "aggregate DOF-updates/s per RK stage, batched uneven periodic vortex cases",
        "value": dof / (t64 / 4), "unit": "DOF-updates/s", "n_gpus": 1, "steps": K, "warmup": W,
        "ms_per_step": t64 * 1e3, "higher_is_better": True, "dtype": "f64", "data": "synthetic",
        "config": {"workload": f"batch_{n_cases}_vortex_cases_n8-{args.batch_max_n}_p1-4_legendre_roe_rk4_cfl0.1-0.04",
                   "seed": args.seed, "cases": n_cases, "elements": int(sum(n ** 3 for n, *_ in cases)),
                   "dof": int(dof), "orders": {str(q): sum(1 for c in cases if c[1] == q) for q in range(1, 5)}},
        "sequential_ms_per_step": t_seq * 1e3, "speedup_vs_sequential": t_seq / t64,
        "groups": {k: groups_of(k) for k in tunings},
        "max_rel_diff_vs_sequential": same,
        "fp32_form": {"value": dof / (t32 / 4), "ms_per_step": t32 * 1e3, "speedup_vs_fp64": t64 / t32,
                      "rho_l2_error_ratio_vs_fp64": {"median": float(np.median(ratio)), "max": float(np.max(ratio)),
                                                     "min": float(np.min(ratio))},
                      "state_max_rel_diff_vs_fp64": {"median": float(np.median(d32)), "max": float(np.max(d32))}},
        "bf16_form": {"value": dof / (tb / 4), "ms_per_step": tb * 1e3, "speedup_vs_fp64": t64 / tb,
                      "rho_l2_error_ratio_vs_fp64": {"median": float(np.median(ratio_b)),
                                                     "max": float(np.max(ratio_b)), "min": float(np.min(ratio_b))},
                      "state_max_rel_diff_vs_fp64": {"median": float(np.median(db)), "max": float(np.max(db))}},
        "rho_l2_error_fp64": {"median": float(np.median(e64)), "max": float(np.max(e64)),
                              "min": float(np.min(e64))},
    }
    print(json.dumps(out))


def tgv_bench(args):
    """The large single case: ne^3 periodic cube [0, 2 pi]^3 (ne = args.tgv,
    96 in the configuration: 110.6M DOF x 5), LegendreHex p = 4, Roe flux,
    inviscid Taylor-Green vortex at Mach 0.1, RK4 to t = 1 at CFL 0.03 (p = 4
    RK4 on this flow is unstable at CFL 0.04: the oracle's run on a 6^3 box
    blows up within 100 steps, and is stable at 0.03 and 0.02), in the plain
    FP64 form and the FP32 form (FP32 contractions and fluxes, compensated
    FP64 solution update).  Reported per form: the stage rate, the fraction
    of the HBM roofline (170 B per DOF per stage), the total mass and kinetic
    energy at 11 times, their drift from t = 0, and FP32 against FP64 at each
    time.  The CPU-baseline leg runs the oracle on an 8^3 box of the same
    case, timing it and comparing both forms' states after the same steps."""
    import numpy as np
    import dg_amd
    from dg_amd import hip

    ne, p, cfl = args.tgv, 4, 0.03
    E, nb = ne ** 3, (p + 1) ** 3
    dof = E * nb
    log = lambda m: print(m, file=sys.stderr, flush=True)       # progress lines

    def toml(n, prec):
        return dg_amd.case_toml(order=p, basis="LegendreHex", flux="Roe", nelem=(n, n, n), lower=(0., 0., 0.),
                                upper=(2 * np.pi,) * 3, stepper="RK4", cfl=cfl, end=1.0, ic="TaylorGreen",
                                ic_data=(0.1,), precision=prec)

    stream = hip.Stream()
    forms = {}
    for form, prec in (("fp64", None), ("fp32", "FP32")):
        s = dg_amd.Solver(toml(ne, prec))
        s.set_stream(stream.handle)
        s.init_state_from_fcn()
        dt, n = s.timestep, s.num_iterations
        I = [s.integrals()]
        times = [0.0]
        ms = 0.0
        bounds = [round(n * k / 10) for k in range(11)]
        for k in range(10):
            ev0, ev1 = hip.Event(), hip.Event()
            ev0.record(stream)
            s.take_time_step(dt, bounds[k + 1] - bounds[k])
            ev1.record(stream)
            ev1.synchronize()
            ms += ev0.elapsed_ms(ev1)
            I.append(s.integrals())
            times.append(s.time)
            log(f"tgv {form}: step {bounds[k + 1]} / {n}, t = {s.time:.4f}, KE = {I[-1][5]:.10e}")
        I = np.array(I)
        t_stage = ms / n / 4 * 1e-3
        forms[form] = {"steps": n, "dt": dt, "t_end": s.time, "ms_per_step": ms / n,
                       "value": dof / t_stage, "finite": bool(np.all(np.isfinite(I))),
                       "roofline_frac": 170.0 * dof / t_stage / 1e9 / HBM_PEAK_GBS,
                       "times": times, "mass": [float(x) for x in I[:, 0]],
                       "kinetic_energy": [float(x) for x in I[:, 5]],
                       "mass_drift": float(np.max(np.abs(I[:, 0] - I[0, 0])) / I[0, 0]),
                       "energy_drift": float(np.max(np.abs(I[:, 4] - I[0, 4])) / I[0, 4]),
                       "kinetic_energy_change": float((I[-1, 5] - I[0, 5]) / I[0, 5])}
        s.close()
    f64, f32 = forms["fp64"], forms["fp32"]
    k64, k32 = np.array(f64["kinetic_energy"]), np.array(f32["kinetic_energy"])
    m64, m32 = np.array(f64["mass"]), np.array(f32["mass"])
    out = {
        "metric": "DOF-updates/s per RK stage, Taylor-Green p=4 to t=1; KE and mass drift FP32 vs FP64",
        "value": f64["value"], "unit": "DOF-updates/s", "n_gpus": 1, "higher_is_better": True,
        "dtype": "f64", "data": "synthetic (Taylor-Green vortex, generated on the GPU)",
        "config": {"workload": f"euler3d_taylor_green_{ne}^3_p4_legendre_roe_rk4_cfl{cfl}_mach0.1_t1",
                   "elements": E, "order": p, "dof": dof},
        "fp64": f64, "fp32_compensated": f32,
        "fp32_vs_fp64": {"speedup": f64["ms_per_step"] / f32["ms_per_step"],
                         "kinetic_energy_max_rel_diff": float(np.max(np.abs(k32 - k64)) / k64[0]),
                         "mass_max_rel_diff": float(np.max(np.abs(m32 - m64)) / m64[0])},
    }
    stream.destroy()
    if not args.no_cpu:
        out["cpu_baseline"], out["oracle_check_8cube"] = tgv_cpu_baseline(toml)
    print(json.dumps(out))


def tgv_cpu_baseline(toml, ne=8, steps=60):
    """CPU leg of the Taylor-Green workload: the oracle on an ne^3 box of the
    same case (p = 4), `steps` RK4 steps timed; both GPU forms run the same
    steps from the same state and are compared with it."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import numpy as np
    import dg_amd
    import oracle as O
    U1, U0, dt = {}, None, None
    for form, prec in (("fp64", None), ("fp32", "FP32")):
        with dg_amd.Solver(toml(ne, prec)) as g:
            g.init_state_from_fcn()
            U0, dt = g.get_state(), g.timestep
            g.take_time_step(dt, steps)
            U1[form] = g.get_state()
    o = O.Solver(O.make_params(order=4, basis="LegendreHex", flux="Roe", nelem=(ne, ne, ne), lo=(0, 0, 0),
                               hi=(2 * np.pi,) * 3, ic="TaylorGreen", ic_data=(0.1,)))
    o.set_state(U0)
    t0 = time.perf_counter()
    o.step("RK4", dt, steps)
    el = time.perf_counter() - t0
    ref = o.get_state()
    scale = float(np.max(np.abs(ref)))
    threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
    dofs = ne ** 3 * 125
    base = {"value": dofs * 4 * steps / el, "unit": "DOF-updates/s", "cores": threads, "kind": "port",
            "cpu_model": cpu_model(),
            "sample": f"oracle on {ne}^3 elements of the same case (p=4, Roe, RK4), {steps} steps in {el:.1f} s"}
    check = {"workload": f"{steps} RK4 steps of the case on {ne}^3 from the same state",
             **{form: {"max_rel_diff": float(np.max(np.abs(U - ref)) / scale)} for form, U in U1.items()}}
    return base, check


def closure_timing(args):
    """Cost of the closure's corrected RK4 step against the plain p = 1 step
    on an n^3 periodic box (n = args.closure_timing; the z-extruded vortex,
    LegendreHex, Roe, RK4 at CFL 0.1), the network at its initial weights
    (the cost does not depend on their values; bound off), and the network
    kernel alone (dg_mlp_forward) on the n^3 feature rows.  One JSON line."""
    import dg_amd
    from dg_amd import closure, hip

    n = args.closure_timing
    K, W = args.steps, args.warmup
    m = closure.MLP(0)
    toml = case_toml(n, p=1)
    res = {}
    with dg_amd.Solver(toml) as s:
        s.init_state_from_fcn()
        E = s.shape[0]
        for name, fn in (("plain", lambda k: s.take_time_step(0.0, k)),
                         ("closure", lambda k: closure.step(s, m, 1e30, k))):
            fn(W)
            hip.synchronize()
            t0 = time.perf_counter()
            fn(K)
            hip.synchronize()
            res[name] = (time.perf_counter() - t0) / K
        X = closure.features(s, s.state_device_ptr())
        m.forward(X, E)
        reps = max(K, 10)
        t0 = time.perf_counter()
        for _ in range(reps):
            m.forward(X, E)
        t_net = (time.perf_counter() - t0) / reps
    m.close()
    flops = 2.0 * (70 * 128 + 128 * 128 + 128 * 40) * E
    print(json.dumps({"metric": "closure step cost", "config": {"workload": f"closure_timing_{n}^3_p1",
                                                                 "elements": E, "steps": K, "warmup": W},
                      "ms_per_rk4_step": {"plain_p1": res["plain"] * 1e3, "closure": res["closure"] * 1e3},
                      "closure_over_plain": res["closure"] / res["plain"],
                      "network_forward": {"ms": t_net * 1e3, "rows": E, "tflops_bf16_incl_sync": flops / t_net / 1e12}}))


def closure_bench(args):
    """Learned closure (coarse p = 1 on a 32^3 periodic box): training rows
    along coarse runs beside FP64 p = 4 runs of seeded vortex /
    acoustic-pulse mixtures (two rollout-training rounds, relaxation time 4
    coarse steps), the network trained by the library's own kernels; then
    held-out seeds run to t = 0.5 with plain p = 1, p = 1 with the closure
    (no bound, and the fallback at 2x the targets' RMS element norm), plain
    p = 2 and p = 3, each compared with the p = 4 run projected to p = 1.
    One JSON line."""
    import numpy as np
    from dg_amd import closure, hip

    n = args.closure
    t0 = time.perf_counter()
    train_seeds = list(range(1000, 1000 + args.closure_seeds))
    log = lambda s: print(s, file=sys.stderr, flush=True)     # progress lines
    # element subsampling keeps each rollout round within 64 M rows (28 GB)
    stride = 1
    while closure.rollout_rows(len(train_seeds), n, 24, stride) > 64 * 2 ** 20 and (n ** 3) % (2 * stride) == 0:
        stride *= 2
    m, hist, rows = closure.train_rollouts(train_seeds, n, fine_order=4, steps=24, tau_steps=4.0,
                                           epochs=args.closure_epochs, bound=2.0, log=log, stride=stride,
                                           rounds=args.closure_rounds, noise=args.closure_noise)
    t_fit = time.perf_counter() - t0
    log(f"training done in {t_fit:.1f} s ({rows} rows, element stride {stride})")
    # a priori: held-out rows along plain coarse runs, network vs the zero correction
    Xv, Yv, rv = closure.generate_rollout([1, 2, 3, 4], n, fine_order=4, steps=24, tau_steps=4.0)
    mse_net, mse_zero = closure.a_priori(m, Xv, Yv, rv)
    Xv.free()
    Yv.free()
    bounds, relax = (None, 2.0), (1.0,)
    log("evaluating held-out seeds")
    ev = closure.evaluate(m, [1, 2, 3, 4], n, 0.5, fine_order=4, bounds=bounds, relax=relax, compare_orders=(2, 3))
    mean = lambda k: float(np.mean([r[k] for r in ev]))
    keys = [("closure" if b is None else f"closure_b{b:g}") + ("" if a == 1.0 else f"_r{a:g}")
            for b in bounds for a in relax]
    out = {
        "metric": "coarse p=1 density L2 error vs the p=4 run projected to p=1, held-out seeds, t = 0.5",
        "config": {"workload": f"closure_{n}^3_p1_mlp70-128-128-40_bf16", "train_seeds": len(train_seeds),
                   "rows": int(rows), "element_stride": stride, "epochs": args.closure_epochs,
                   "rollout_rounds": args.closure_rounds, "feature_jitter": args.closure_noise},
        "train_s": t_fit, "loss_history": hist,
        "target_rms_element_norm": m.target_rms,
        "a_priori_heldout_mse": {"network": mse_net, "zero_correction": mse_zero,
                                 "fraction_removed": 1.0 - mse_net / mse_zero},
        "p1_rho_error": mean("p1_rho_error"), "p2_rho_error": mean("p2_rho_error"),
        "p3_rho_error": mean("p3_rho_error"),
        "closure": {k: {"rho_error": mean(f"{k}_rho_error"),
                        "error_ratio_vs_p1": mean(f"{k}_rho_error") / mean("p1_rho_error"),
                        "fallback_elements": int(sum(r[f"{k}_fallback_elements"] for r in ev)),
                        "wall_per_time_unit_s": mean(f"{k}_wall_per_time")} for k in keys},
        "wall_per_time_unit_s": {"p1": mean("p1_wall_per_time"), "p2": mean("p2_wall_per_time"),
                                 "p3": mean("p3_wall_per_time"), "p4": mean("fine_wall_per_time")},
        "per_seed": ev,
    }
    m.close()
    print(json.dumps(out))


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--ne", type=int, default=NE, help=argparse.SUPPRESS)
    # other orders / the warped box: measurements beside the headline line
    ap.add_argument("--order", type=int, default=P, help=argparse.SUPPRESS)
    ap.add_argument("--warp", type=float, default=0.0, help=argparse.SUPPRESS)
    ap.add_argument("--dim", type=int, default=3, choices=(2, 3), help=argparse.SUPPRESS)
    # data.h5 write / read-back of the workload's state (file path)
    ap.add_argument("--io", default=None, help=argparse.SUPPRESS)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    # the FP32 form only (for profiling its kernel); --no-fp32 skips it
    ap.add_argument("--fp32", action="store_true", help=argparse.SUPPRESS)
    ap.add_argument("--no-fp32", action="store_true", help="skip the reduced-precision legs")
    # one form only (for profiling its kernel): FP32, BF16 or BF16x3
    ap.add_argument("--precision", default=None, help=argparse.SUPPRESS)
    # batched uneven cases (dg_batch_*): number of cases and their seed
    ap.add_argument("--batch", type=int, default=0, help=argparse.SUPPRESS)
    ap.add_argument("--seed", type=int, default=7, help=argparse.SUPPRESS)
    ap.add_argument("--batch-max-n", type=int, default=32, help=argparse.SUPPRESS)
    # learned closure: coarse mesh edge, training seeds, epochs
    ap.add_argument("--closure", type=int, default=0, help=argparse.SUPPRESS)
    ap.add_argument("--closure-seeds", type=int, default=16, help=argparse.SUPPRESS)
    ap.add_argument("--closure-epochs", type=int, default=6, help=argparse.SUPPRESS)
    ap.add_argument("--closure-rounds", type=int, default=2, help=argparse.SUPPRESS)
    ap.add_argument("--closure-noise", type=float, default=0.05, help=argparse.SUPPRESS)
    ap.add_argument("--closure-timing", type=int, default=0, help=argparse.SUPPRESS)
    # the large Taylor-Green case (mesh edge; 96 in the configuration)
    ap.add_argument("--tgv", type=int, default=0, help=argparse.SUPPRESS)
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: the path runs on one GPU; --gpus {args.gpus} is not supported "
              "(the path is measured at one GPU's real shape)", file=sys.stderr)
        sys.exit(2)

    import numpy as np
    import dg_amd
    from dg_amd import hip

    assert hip.device_count() > 0, "bench.py needs a GPU"
    if args.batch:
        batch_bench(args)
        return
    if args.closure:
        closure_bench(args)
        return
    if args.closure_timing:
        closure_timing(args)
        return
    if args.tgv:
        tgv_bench(args)
        return
    ne, order, dim = args.ne, args.order, args.dim
    if dim == 2 and ne == NE:
        ne = 1024                         # 2D: 1024^2 elements, the DOF count of the 3D headline at p=3
    stream = hip.Stream()                 # default priority
    E = ne ** dim
    nb = (order + 1) ** dim
    nvar = dim + 2
    dof = E * nb

    def timed_run(precision):
        """Warm-up and timed RK4 steps; (solver, ms per step, wall s)."""
        s = dg_amd.Solver(case_toml(ne, order, warp=args.warp, dim=dim, precision=precision))
        s.set_stream(stream.handle)
        s.init_state_from_fcn()
        dt = s.timestep
        s.take_time_step(dt, args.warmup)
        hip.synchronize()
        ev0, ev1 = hip.Event(), hip.Event()
        t0 = time.perf_counter()
        ev0.record(stream)
        s.take_time_step(dt, args.steps)      # 4 stages per step, all launches on `stream`
        ev1.record(stream)
        ev1.synchronize()
        hip.synchronize()
        return s, ev0.elapsed_ms(ev1) / args.steps, time.perf_counter() - t0

    if args.io:
        s = dg_amd.Solver(case_toml(ne, order, warp=args.warp, dim=dim))
        s.init_state_from_fcn()
        io_bench(s, args.io)
        return
    s, ms_per_step, wall = timed_run(args.precision or ("FP32" if args.fp32 else None))
    dt = s.timestep
    t_stage = ms_per_step / 4 * 1e-3
    value = dof / t_stage
    headline = dim == 3 and not args.warp and order == P and ne == NE

    def to_acc_steps(sv):
        # the configuration's 50 RK4 steps in all (warm-up and timed steps count)
        done = args.warmup + args.steps
        if done < ACC_STEPS:
            sv.take_time_step(sv.timestep, ACC_STEPS - done)
        return max(done, ACC_STEPS)

    nacc = to_acc_steps(s)
    # accuracy of the run: L2 error vs the exact advected vortex after nacc steps
    err = s.get_error()
    finite = bool(np.all(np.isfinite(err)))

    bytes_stage = ALG_BYTES_PER_DOF * nvar / 5 * dof
    achieved = bytes_stage / t_stage / 1e9
    flops_stage = alg_flops_per_element(order) * E if dim == 3 else None
    precision = args.precision or ("FP32" if args.fp32 else None)
    name, per_stage = stage_kernels(order, E, dim, args.warp, precision)
    out = {
        "metric": METRIC,
        "value": value,
        "unit": "DOF-updates/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": (precision or "f64").lower(),
        "data": "synthetic (z-extruded isentropic vortex, generated on the GPU)" if dim == 3 else
                "synthetic (2D isentropic vortex, generated on the GPU)",
        "config": {"workload": (f"euler3d_periodic_box_{ne}^3_p{order}_legendre_roe_rk4_cfl0.1"
                                + (f"_warp{args.warp}" if args.warp else "")) if dim == 3 else
                   f"euler2d_periodic_box_{ne}^2_p{order}_legendre_roe_rk4_cfl0.1",
                   "elements": E, "order": order, "dof": dof, "variables": nvar, "flux": "Roe",
                   "basis": "LegendreHex" if dim == 3 else "LegendreQuad", "stepper": "RK4", "dt": dt,
                   "domain": "[-5,5]^3" if dim == 3 else "[-5,5]^2"},
        "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS,
                     "traffic": measured_traffic() if headline else None},
        "kernel": {"name": name, "launches_per_stage": per_stage, "launches": 4 * per_stage * args.steps,
                   "avg_stage_ms": ms_per_step / 4,
                   "alg_bytes_per_stage": bytes_stage, "alg_flops_per_stage": flops_stage,
                   "fp64_tflops": flops_stage / t_stage / 1e12 if flops_stage else None,
                   "fp64_frac": flops_stage / t_stage / 1e12 / FP64_PEAK_TFLOPS if flops_stage else None},
        "l2_error_vs_exact": [float(x) for x in err],
        "l2_error_steps": nacc,
        "finite": finite,
        "wall_s": wall,
    }
    if headline:
        # the second denominator: the copy rate a plain kernel reaches on this GPU
        copy = measured_copy_gbs()
        out["roofline"]["copy_measured_GBps"] = copy
        out["roofline"]["frac_vs_copy"] = achieved / copy if copy else None
    gpu_step = None
    if dim == 3 and not args.warp and not args.fp32 and not args.precision and not args.no_fp32:
        # the reduced-precision forms on the same workload, against this FP64
        # run: FP32 (contractions and fluxes on the VALU), BF16 and BF16x3
        # (the FP32 form with the x-y projection on bf16 matrix cores: one
        # bf16 term / a hi-lo split with three products); all keep FP64 RK
        # registers with the compensated update, M^-1 and reductions
        U64 = s.get_state()
        s.close()
        for key, prec, what in (("fp32_form", "FP32", "f32 traces/fluxes/contractions"),
                                ("bf16x3_form", "BF16x3", "f32, x-y projection as bf16 hi/lo MFMA (3 products)"),
                                ("bf16_form", "BF16", "f32, x-y projection as bf16 MFMA")):
            sr, msr, _ = timed_run(prec)
            to_acc_steps(sr)
            errr = sr.get_error()
            Ur = sr.get_state()
            diff = float(np.max(np.abs(Ur - U64)) / np.max(np.abs(U64)))
            del Ur
            out[key] = {
                "value": dof / (msr / 4 * 1e-3), "unit": "DOF-updates/s", "ms_per_step": msr,
                "speedup_vs_fp64": ms_per_step / msr,
                "dtype": what + ", f64 RK registers (compensated update), M^-1 and reductions",
                "kernel": stage_kernels(order, E, dim, args.warp, prec)[0],
                "l2_error_vs_exact": [float(x) for x in errr],
                # the extruded vortex has w = 0 exactly: FP64 keeps it at round-off (~1e-16) and
                # FP32 at ~1e-8, so the ratio is reported for the variables with a real error
                "l2_error_ratio_vs_fp64": [float(a / b) if b > 1e-12 else None for a, b in zip(errr, err)],
                "state_max_rel_diff_vs_fp64": diff,
            }
            sr.close()
        del U64
    else:
        s.close()
    if headline and not args.fp32 and not args.precision and not args.no_fp32:
        # the second input of the configuration: a Gaussian density bump
        # (amplitude 0.2, width 1) in uniform flow of speed 1 along a seeded
        # random direction (numpy default_rng(2024), a normalised Gaussian
        # vector), p = 1, both forms, 50 steps; L2 error vs exact advection.
        # CFL 0.06: at this Mach number (0.85) p = 3 RK4 is unstable at 0.1
        # (the oracle blows up as well)
        v = np.random.default_rng(2024).standard_normal(3)
        v /= np.linalg.norm(v)
        bump = {"data": [0.2, 1.0, float(v[0]), float(v[1]), float(v[2]), 1.0, 0.0, 0.0, 0.0], "cfl": 0.06}
        for form, prec in (("fp64", None), ("fp32", "FP32")):
            sb = dg_amd.Solver(dg_amd.case_toml(order=P, basis="LegendreHex", flux="Roe", nelem=(ne, ne, ne),
                                                lower=(-5., -5., -5.), upper=(5., 5., 5.), stepper="RK4", cfl=0.06,
                                                end=1.0, ic="GaussianBump", ic_data=bump["data"], precision=prec))
            sb.set_stream(stream.handle)
            sb.init_state_from_fcn()
            e0 = sb.get_error()
            ev0, ev1 = hip.Event(), hip.Event()
            ev0.record(stream)
            sb.take_time_step(sb.timestep, ACC_STEPS)
            ev1.record(stream)
            ev1.synchronize()
            bump[form] = {"ms_per_step": ev0.elapsed_ms(ev1) / ACC_STEPS,
                          "value": dof / (ev0.elapsed_ms(ev1) / ACC_STEPS / 4 * 1e-3),
                          "l2_error_vs_exact_t0": [float(x) for x in e0],
                          "l2_error_vs_exact": [float(x) for x in sb.get_error()], "steps": ACC_STEPS}
            sb.close()
        bump["l2_error_ratio_fp32_vs_fp64"] = [float(a / b) for a, b in zip(bump["fp32"]["l2_error_vs_exact"],
                                                                          bump["fp64"]["l2_error_vs_exact"])]
        out["gaussian_bump"] = bump
    if headline and not args.no_cpu:
        # one RK4 step of both forms on the oracle's box, compared by the
        # CPU-baseline leg with the oracle's step from the same state
        U1 = {}
        for form, prec in (("fp64", None), ("fp32", "FP32")):
            so = dg_amd.Solver(case_toml(ORACLE_NE, P, precision=prec))
            so.init_state_from_fcn()
            U0o, dto = so.get_state(), so.timestep
            so.take_time_step(dto, 1)
            U1[form] = so.get_state()
            so.close()
        gpu_step = (U0o, dto, U1)
    stream.destroy()
    if not args.no_cpu and dim == 3:
        out["cpu_baseline"], check = cpu_baseline(gpu_step)
        if check is not None:
            out["l2_err_vs_fp64_oracle"] = check
    else:
        out["cpu_baseline"] = None
    print(json.dumps(out))


if __name__ == "__main__":
    main()
