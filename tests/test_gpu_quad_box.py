"""2D boxes large enough for the 16-elements-a-wave stage kernel: residual, one
RK4 and one forward-Euler step against the 2D oracle.  Element counts just
above the size where it takes over, with remainders of 16 and of the 8 XCDs'
shares among them, and single-element directions (an element that is its own
neighbour); all orders, bases and fluxes."""
import numpy as np
import pytest

import dg2d
import dg_amd
from dg_amd import hip

pytestmark = pytest.mark.gpu

# order, elements: the kernel takes over at 768, 2048, 3072, 2304, 2560 elements
CASES = [
    (1, (32, 24), "LegendreQuad", "Roe"), (1, (1, 769), "LagrangeQuad", "HLLC"), (1, (29, 31), "LegendreQuad", "LaxFriedrichs"),
    (2, (32, 64), "LegendreQuad", "HLLC"), (2, (2063, 1), "LagrangeQuad", "Roe"), (2, (45, 47), "LagrangeQuad", "LaxFriedrichs"),
    (3, (48, 64), "LagrangeQuad", "LaxFriedrichs"), (3, (55, 57), "LegendreQuad", "Roe"), (3, (3, 1025), "LegendreQuad", "HLLC"),
    (4, (48, 48), "LegendreQuad", "Roe"), (4, (2, 1153), "LagrangeQuad", "HLLC"),
    (5, (51, 51), "LagrangeQuad", "Roe"), (5, (40, 64), "LegendreQuad", "LaxFriedrichs"),
]


@pytest.mark.parametrize("order,ne,basis,flux", CASES)
def test_against_the_oracle(order, ne, basis, flux):
    print(f"quad box p={order} {ne} {basis} {flux}", flush=True)
    lo, hi, data = (-5., -4.), (6., 4.), (1.0, 0.7, -0.4, 1.0, 3.0)
    dt = 0.02 / max(ne) / (2 * order + 1)
    eps, growth = 2.0 ** -53, (2 * order + 1) ** 2
    for stepper in ("RK4", "FE"):
        g = dg_amd.Solver(dg_amd.case_toml(order=order, basis=basis, flux=flux, nelem=ne, lower=lo, upper=hi,
                                           stepper=stepper, timestep=dt, ic="IsentropicVortex", ic_data=data))
        o = dg2d.Box2D(order, basis, flux, ne, lo, hi, ic="IsentropicVortex", ic_data=data)
        with g:
            g.init_state_from_fcn()
            U0 = g.get_state()
            u, r = hip.Buffer.from_array(U0), hip.Buffer(U0.size)
            g.get_residual(u.addr, r.addr)
            hip.synchronize()
            R = r.download(U0.shape)
            g.take_time_step()
            U1 = g.get_state()
            u.free()
            r.free()
        ref = o.residual(U0)
        # the residual is a difference of sums of some hundred rounded
        # operations on terms of the fluxes' size; the flux terms are at most
        # the states' scale (5) times the larger face length
        size = 5. * np.max(np.abs(U0)) * max((hi[0] - lo[0]) / ne[0], (hi[1] - lo[1]) / ne[1])
        assert np.max(np.abs(R - ref)) <= 256 * eps * (np.max(np.abs(ref)) + size)
        o.U = U0.copy()
        o.step(stepper, dt, 1)
        # a step's increment is dt M^-1 of it, with M^-1 growing as
        # (2 p + 1)^2 over the element's area; the state adds its last place
        jdet = (hi[0] - lo[0]) * (hi[1] - lo[1]) / (4. * ne[0] * ne[1])
        tol = 256 * eps * growth * dt / jdet * (np.max(np.abs(ref)) + size) + 4 * 2.0 ** -52 * np.max(np.abs(U0))
        assert np.all(np.isfinite(U1)) and np.max(np.abs(U1 - U0)) > 0.0
        assert np.max(np.abs(U1 - o.U)) <= tol, (stepper, np.max(np.abs(U1 - o.U)), tol)
