"""Boxes of a few elements per CU, whose FP64 stage runs the face and the
volume term in two halves of a workgroup: the residual and one RK4 and one
forward-Euler step against the oracle, on both sides of the sizes where that
ends (p = 1: 2048 elements, p = 2: 1024, p = 3: 512 and 768), single elements
among them.  The steps' arithmetic is the whole workgroup's, so the bars are
test_gpu_parity.py's: 1e-12 relative.  On top comes what the oracle's element
widths carry, differences of node coordinates up to the number n of unit
elements in a row: n eps of each face's flux (about 4, six faces) in a
residual that is what the fluxes leave."""
import numpy as np
import pytest

import dg_amd
import oracle as O
from dg_amd import hip

pytestmark = pytest.mark.gpu

CASES = [(1, (1, 1, 1), "LagrangeHex", "HLLC"), (1, (16, 16, 8), "LegendreHex", "Roe"),
         (1, (3, 683, 1), "LegendreHex", "LaxFriedrichs"), (2, (8, 8, 16), "LagrangeHex", "Roe"),
         (2, (25, 41, 1), "LegendreHex", "HLLC"), (2, (1, 2, 1), "LegendreHex", "LaxFriedrichs"),
         (3, (8, 8, 8), "LagrangeHex", "HLLC"), (3, (27, 19, 1), "LegendreHex", "Roe"),
         (3, (8, 8, 12), "LegendreHex", "LaxFriedrichs"), (3, (769, 1, 1), "LagrangeHex", "Roe"),
         (3, (1, 1, 2), "LegendreHex", "Roe")]


def relerr(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


@pytest.mark.parametrize("order,ne,basis,flux", CASES)
def test_small_box(order, ne, basis, flux):
    print(f"small box p={order} {ne} {basis} {flux}", flush=True)
    lo, hi, dt = (0., 0., 0.), tuple(float(n) for n in ne), 0.01
    data = (0.2, 1.5, 0.6, -0.48, 0.64, 1.0, 0.4, 0.5, 0.6)
    for stepper in ("RK4", "FE"):
        g = dg_amd.Solver(dg_amd.case_toml(order=order, basis=basis, flux=flux, nelem=ne, lower=lo, upper=hi,
                                           stepper=stepper, timestep=dt, ic="GaussianBump", ic_data=data))
        o = O.Solver(O.make_params(order=order, basis=basis, flux=flux, nelem=ne, lo=lo, hi=hi, gamma=1.4, R=1.0,
                                   ic="GaussianBump", ic_data=data))
        with g:
            o.init_state()
            # every coefficient exercised, elements unlike their neighbours
            U = o.get_state()
            U = U * (1.0 + 1e-3 * np.random.default_rng(7).standard_normal(U.shape))
            g.set_state(U)
            o.set_state(U)
            u, r = hip.Buffer.from_array(U), hip.Buffer(U.size)
            g.get_residual(u.addr, r.addr)
            hip.synchronize()
            R = o.residual(U)
            bar = 1e-12 + max(ne) * np.finfo(float).eps * 24.0 / np.max(np.abs(R))
            assert relerr(r.download(U.shape), R) < bar
            g.take_time_step(0.0, 1)
            o.step(stepper, dt, 1)
            assert relerr(g.get_state(), o.get_state()) < 1e-12
            u.free()
            r.free()
