"""Boxes large enough for the two-pass RK stage (faces once, then the
elements): one RK4 and one forward-Euler step against the steps composed from
the residual and inverse-mass calls, which run the fused kernel on the same
state.  Element counts just above the size where the two passes take over
(and one below), with every remainder of the workgroups' element counts among
them, single-element directions (an element that is its own neighbour), all
orders, bases and fluxes."""
import numpy as np
import pytest

import dg_amd
from dg_amd import hip

pytestmark = pytest.mark.gpu

# order, elements: in FP64 p = 1 takes over at 4608 elements, p = 2 at 2560,
# the rest at 2816, in the FP32 form at 7168, 5120, 5120, 24576, 6656;
# the workgroups of the two passes hold 7 and 6, 5 and 4, 4 and 5, 3 and 3,
# 3 and 2 elements
CASES = [
    (1, (17, 17, 16), "LegendreHex", "Roe"), (1, (19, 16, 25), "LagrangeHex", "HLLC"),
    (2, (14, 15, 13), "LagrangeHex", "LaxFriedrichs"), (2, (17, 19, 17), "LegendreHex", "Roe"),
    (2, (1, 2561, 1), "LegendreHex", "HLLC"),
    (3, (17, 13, 13), "LegendreHex", "Roe"), (3, (2819, 1, 1), "LagrangeHex", "HLLC"),
    (3, (14, 14, 14), "LegendreHex", "LaxFriedrichs"), (3, (18, 18, 18), "LagrangeHex", "Roe"),
    (3, (19, 17, 17), "LegendreHex", "HLLC"), (3, (1, 32, 161), "LegendreHex", "LaxFriedrichs"),
    (4, (15, 14, 14), "LegendreHex", "HLLC"), (4, (23, 22, 23), "LagrangeHex", "Roe"),
    (4, (30, 29, 29), "LegendreHex", "LaxFriedrichs"),
    (5, (15, 15, 13), "LegendreHex", "Roe"), (5, (19, 19, 19), "LagrangeHex", "LaxFriedrichs"),
]


def solver(order, ne, basis, flux, stepper="RK4", precision=None):
    dt = 0.02 / max(ne) / (2 * order + 1)
    # unequal element widths; the vortex stays resolved by the small boxes
    s = dg_amd.Solver(dg_amd.case_toml(order=order, basis=basis, flux=flux, nelem=ne, lower=(-5., -4., -3.),
                                       upper=(5., 4., 3.), stepper=stepper, timestep=dt, precision=precision,
                                       ic="ExtrudedIsentropicVortex", ic_data=(1.0, 0.7, -0.4, 1.0, 3.0, 0.3, -0.2)))
    s.init_state_from_fcn()
    return s, dt


def composed(s, U0, dt, stepper):
    """a step from get_residual and mult_inv_mass_matrix on buffers of the host's own"""
    n = U0.size
    u, r, st = hip.Buffer(n), hip.Buffer(n), hip.Stream()      # a stream of its own: the fused kernel

    def tendency(U):
        u.upload(U)
        s.get_residual(u.addr, r.addr, st.h.value)
        s.mult_inv_mass_matrix(dt, r.addr, r.addr, st.h.value)
        hip.synchronize()
        return r.download(U.shape)

    k1 = tendency(U0)
    if stepper == "FE":
        out = U0 + k1
    else:
        k2 = tendency(U0 + 0.5 * k1)
        k3 = tendency(U0 + 0.5 * k2)
        k4 = tendency(U0 + k3)
        out = U0 + (k1 + 2.0 * k2 + 2.0 * k3 + k4) / 6.0
    u.free()
    r.free()
    return out


@pytest.mark.parametrize("order,ne,basis,flux", CASES)
@pytest.mark.parametrize("precision", [None, "FP32"])
def test_step_matches_the_composed_step(order, ne, basis, flux, precision):
    print(f"two-pass p={order} {ne} {basis} {flux} {precision}", flush=True)
    for stepper in ("RK4", "FE"):
        s, dt = solver(order, ne, basis, flux, stepper, precision)
        with s:
            U0 = s.get_state()
            s.take_time_step()
            U1 = s.get_state()
            ref = composed(s, U0, dt, stepper)
        d = np.max(np.abs(U1 - ref))
        # the increment carries the form's rounding: 2^-53 (2^-24) per
        # operation over some hundreds of operations and the growth of M^-1,
        # (2 p + 1)^3 between the modes; the state adds its own last place
        inc = np.max(np.abs(ref - U0))
        eps = 2.0 ** -53 if precision is None else 2.0 ** -24
        tol = 64 * eps * (2 * order + 1) ** 3 * inc + 4 * 2.0 ** -52 * np.max(np.abs(ref))
        assert np.all(np.isfinite(U1)) and inc > 0.0
        assert d <= tol, (stepper, d, tol, inc)


@pytest.mark.parametrize("order,ne,basis,flux", CASES)
@pytest.mark.parametrize("precision", [None, "FP32"])
def test_residual_matches_the_fused_kernel(order, ne, basis, flux, precision):
    """on the handle's stream, against the fused kernel on the caller's"""
    print(f"two-pass residual p={order} {ne} {basis} {flux} {precision}", flush=True)
    s, _ = solver(order, ne, basis, flux, "RK4", precision)
    with s:
        U = s.get_state()
        u, ra, rb, st = hip.Buffer.from_array(U), hip.Buffer(U.size), hip.Buffer(U.size), hip.Stream()
        s.get_residual(u.addr, ra.addr)
        s.get_residual(u.addr, rb.addr, st.h.value)
        hip.synchronize()
        a, b = ra.download(U.shape), rb.download(U.shape)
        for buf in (u, ra, rb):
            buf.free()
    # differences of sums of some hundred rounded operations on flux terms
    # of at most the states' scale (5) times the largest face
    h = sorted((hi - lo) / n for lo, hi, n in zip((-5., -4., -3.), (5., 4., 3.), ne))
    size = 5. * np.max(np.abs(U)) * h[1] * h[2]
    eps = 2.0 ** -53 if precision is None else 2.0 ** -24
    assert np.all(np.isfinite(a)) and np.max(np.abs(b)) > 0.0
    assert np.max(np.abs(a - b)) <= 64 * eps * (np.max(np.abs(b)) + size)


@pytest.mark.parametrize("precision", [None, "FP32"])
def test_integrals_are_conserved(precision):
    s, _ = solver(3, (18, 18, 18), "LegendreHex", "Roe", "RK4", precision)
    with s:
        I0 = s.integrals()
        s.take_time_step(0.0, 20)
        I1 = s.integrals()
    bar = 1e-13 if precision is None else 1e-6
    assert np.max(np.abs(I1[:5] - I0[:5])) <= bar * np.max(np.abs(I0[:5]))


def test_closure_step_with_a_zero_network_is_the_plain_step():
    from dg_amd import closure
    m = closure.MLP(0)
    p = m.params()
    p[:] = 0.0
    m.set_params(p)
    a, _ = solver(1, (17, 17, 16), "LegendreHex", "Roe")
    b, _ = solver(1, (17, 17, 16), "LegendreHex", "Roe")
    with a, b:
        a.take_time_step(0.0, 2)
        closure.step(b, m, 1e30, 2)
        Ua, Ub = a.get_state(), b.get_state()
    m.close()
    assert np.max(np.abs(Ua - Ub)) <= 4 * 2.0 ** -52 * np.max(np.abs(Ua))


# cases of one batch: every order's group (and one in the FP32 form) is large
# enough together, though no case is by itself; uneven sizes, so that the
# workgroups' sequences end in every remainder, and single-element cases
BATCH = [
    (1, (13, 11, 17), "LegendreHex", "Roe", None), (1, (17, 17, 8), "LegendreHex", "Roe", None),
    (2, (9, 9, 9), "LagrangeHex", "HLLC", None), (2, (13, 7, 5), "LagrangeHex", "HLLC", None),
    (2, (1, 1, 1), "LagrangeHex", "HLLC", None), (2, (11, 12, 11), "LagrangeHex", "HLLC", None),
    (3, (14, 14, 14), "LegendreHex", "LaxFriedrichs", None), (3, (3, 5, 7), "LegendreHex", "LaxFriedrichs", None),
    (4, (13, 13, 13), "LegendreHex", "Roe", None), (4, (9, 9, 9), "LegendreHex", "Roe", None),
    (5, (12, 12, 12), "LagrangeHex", "Roe", None), (5, (11, 11, 10), "LagrangeHex", "Roe", None),
    (2, (15, 15, 15), "LegendreHex", "Roe", "FP32"), (2, (12, 13, 12), "LegendreHex", "Roe", "FP32"),
]


def test_batch_matches_each_case_alone():
    made = [(solver(o, ne, b, f, "RK4", pr), solver(o, ne, b, f, "RK4", pr)) for o, ne, b, f, pr in BATCH]
    batch_s, solo_s = [m[0][0] for m in made], [m[1][0] for m in made]
    with dg_amd.Batch(batch_s) as batch:
        for n in (1, 2, 7):          # replays of the captured step, then the tuned one
            print(f"two-pass batch, {n} steps", flush=True)
            before = [s.get_state() for s in solo_s]
            for sb, U in zip(batch_s, before):
                sb.set_state(U)
            batch.step(n)
            for (order, ne, _, _, prec), sb, so, U0 in zip(BATCH, batch_s, solo_s, before):
                so.take_time_step(0.0, n)
                ref, U1 = so.get_state(), sb.get_state()
                # as above, over n steps
                inc = np.max(np.abs(ref - U0))
                eps = 2.0 ** -53 if prec is None else 2.0 ** -24
                tol = n * (64 * eps * (2 * order + 1) ** 3 * inc + 4 * 2.0 ** -52 * np.max(np.abs(ref)))
                d = np.max(np.abs(U1 - ref))
                assert np.all(np.isfinite(U1)) and inc > 0.0
                assert d <= tol, (order, ne, prec, n, d, tol)
        for (cap, ncases, elements, ms) in batch.tiles():
            assert min(ms) > 0.0 and cap in (2, 3)
    for s in batch_s + solo_s:
        s.close()
