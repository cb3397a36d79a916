"""The dense inverse mass matrices of trilinear elements, whose columns are
fetched 16 entries at a time, ahead of the residual in a stage: orders with
fewer, as many and more rows than that, single elements and odd counts; and
boxes far from the origin, where the Jacobians must round at the elements'
size.  Bar as in test_gpu_mapped.py: 1e-11 through M^-1; far from the origin
the node coordinates carry 1e3 eps of the element width on both sides, which
the flux differences of the residual raise by about ten."""
import numpy as np
import pytest

import dg_amd
import oracle as O
from dg_amd import hip

pytestmark = pytest.mark.gpu


def pair(order, ne, basis, flux, lo, hi, centre, dt):
    data = (0.2, 1.5, 0.6, -0.48, 0.64, 1.0) + centre
    g = dg_amd.Solver(dg_amd.case_toml(order=order, basis=basis, flux=flux, nelem=ne, lower=lo, upper=hi,
                                       stepper="RK4", timestep=dt, end=1.0, ic="GaussianBump", ic_data=data,
                                       warp=0.1, normals="exact"))
    o = O.Solver(O.make_params(order=order, basis=basis, flux=flux, nelem=ne, lo=lo, hi=hi, gamma=1.4, R=1.0,
                               ic="GaussianBump", ic_data=data, warp=0.1, exact_normals=True))
    return g, o


def relerr(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


@pytest.mark.parametrize("order", [1, 2, 3, 4])
@pytest.mark.parametrize("ne,shift", [((3, 3, 3), 0.0), ((5, 3, 4), 0.0), ((3, 4, 3), 1000.0)])
def test_step_and_inverse_mass(order, ne, shift):
    basis = "LegendreHex" if order % 2 else "LagrangeHex"
    flux = ("LaxFriedrichs", "HLLC", "Roe")[order % 3]
    print(f"dense mass p={order} {ne} {basis} {flux} shift {shift}", flush=True)
    lo = tuple(shift - 0.5 * n for n in ne)
    hi = tuple(shift + 0.5 * n for n in ne)
    dt = 0.002
    g, o = pair(order, ne, basis, flux, lo, hi, (shift, shift, shift), dt)
    with g:
        o.init_state()
        U = o.get_state()
        g.set_state(U)
        R = o.residual(U)
        d, r = hip.Buffer.from_array(R), hip.Buffer(U.size)
        g.mult_inv_mass_matrix(0.37, d.addr, r.addr)
        hip.synchronize()
        assert relerr(r.download(U.shape), o.inv_mass(0.37, R)) < 1e-11
        g.take_time_step(0.0, 3)
        o.step("RK4", dt, 3)
        assert relerr(g.get_state(), o.get_state()) < 1e-11
        d.free()
        r.free()
