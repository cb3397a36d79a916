"""Stepper.compensated where the update runs in the element pass: many small
steps of a box large enough for the two passes, and of a batch that is only as
a group (and of one that is fused), against RK4 with the solution accumulated
in long double (see test_gpu_compensated.py, whose small boxes run the fused
stage)."""
import numpy as np
import pytest

import dg_amd
from test_gpu_compensated import ld_reference, toml

pytestmark = pytest.mark.gpu

# plain rounding is a random walk of 0.29 spacings a step: over 300 steps, 5
# spacings, and some 4 times that at the worst of the 10^5 coefficients
DT, N = 1e-4, 300


def run(ne, comp, batch):
    cases = [dg_amd.Solver(toml(ne, dt=DT, comp=comp)) for _ in range(2 if batch else 1)]
    for s in cases:
        s.init_state_from_fcn()
    U0 = cases[0].get_state()
    if batch:
        with dg_amd.Batch(cases) as b:
            b.step(N)
    else:
        cases[0].take_time_step(DT, N)
    U = [s.get_state() for s in cases]
    for s in cases:
        s.close()
    return U0, U


@pytest.mark.parametrize("ne,batch", [((17, 17, 16), False), ((17, 17, 8), True), ((9, 9, 8), True)])
def test_two_pass_update_tracks_long_double_accumulation(ne, batch):
    print(f"compensated two-pass steps on {ne}, batch: {batch}", flush=True)
    res = {}
    for comp in (False, True):
        U0, res[comp] = run(ne, comp, batch)
    with dg_amd.Solver(toml(ne, dt=DT, comp=False)) as g:
        g.init_state_from_fcn()
        ref = ld_reference(g, U0, DT, N)
    ulp = float(np.spacing(np.max(np.abs(ref.astype(np.float64)))))
    err = {c: max(float(np.max(np.abs(U.astype(np.longdouble) - ref)) / ulp) for U in res[c]) for c in res}
    print(f"distance to the long-double accumulation in spacings: plain {err[False]:.1f}, "
          f"compensated {err[True]:.2f}", flush=True)
    # the bounds of test_gpu_compensated.py
    assert err[True] <= 4.0
    assert err[False] >= 4.0 * max(err[True], 1.0)
