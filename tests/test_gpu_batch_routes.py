"""A batch group of many tiny cases runs the fused stage where a workgroup of
the two passes, which holds elements of one case, would be part empty, and the
two passes where the cases fill it.  The tuner shows the route: the two
passes have one form, whose time stands for every candidate."""
import numpy as np
import pytest

import dg_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,ne,cases,two_pass", [(4, (2, 2, 2), 352, False), (4, (3, 2, 2), 235, True),
                                                     (1, (2, 2, 2), 580, False), (3, (5, 5, 5), 23, True)])
def test_route_of_tiny_cases(order, ne, cases, two_pass):
    print(f"batch of {cases} {ne} p={order}", flush=True)
    toml = dg_amd.case_toml(order=order, basis="LegendreHex", flux="Roe", nelem=ne, timestep=1e-3 / (2 * order + 1),
                            ic="ExtrudedIsentropicVortex", ic_data=(1.0, 0.7, -0.4, 1.0, 3.0))
    made = [dg_amd.Solver(toml) for _ in range(cases)]
    for s in made:
        s.init_state_from_fcn()
    U0 = made[0].get_state()
    with dg_amd.Batch(made) as b:
        b.step(8)
        (_, nc, elements, ms), = b.tiles()
    with dg_amd.Solver(toml) as s:
        s.init_state_from_fcn()
        s.take_time_step(0.0, 8)
        R = s.get_state()
    # round-off of the routes over 8 steps (the bound of test_gpu_two_pass.py)
    inc = np.max(np.abs(R - U0))
    tol = 8 * (64 * 2.0 ** -53 * (2 * order + 1) ** 3 * inc + 4 * 2.0 ** -52 * np.max(np.abs(R)))
    for s in made[:: cases // 8]:
        assert np.max(np.abs(s.get_state() - R)) <= tol
    for s in made:
        s.close()
    assert nc == cases and elements == cases * int(np.prod(ne))
    assert (len(set(ms)) == 1) == two_pass, ms
