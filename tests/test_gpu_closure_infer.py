"""The closure step's network pass, which forms its features from the state,
against the same step composed from the features, forward, residual and
inverse-mass calls: boxes of uneven sizes, with single-element directions,
fewer elements than a wave's 16 rows, remainders of them and of a workgroup's
64 and 128; and the forward pass at row counts on both sides of the line
between the two workgroup sizes (16384 rows)."""
import numpy as np
import pytest

import dg_amd
import mlp as MO
from dg_amd import closure, hip

pytestmark = pytest.mark.gpu


def network(seed=5):
    rng = np.random.default_rng(seed)
    m = closure.MLP(0)
    p = np.concatenate([rng.normal(0, 0.2, int(np.prod(s))) for _, s in MO.SHAPES]).astype(np.float32)
    m.set_params(p)
    m.set_scaling(rng.normal(0, 0.1, MO.NF).astype(np.float32), rng.uniform(0.5, 2.0, MO.NF).astype(np.float32),
                  rng.uniform(0.5, 2.0, MO.NO).astype(np.float32))
    return m


@pytest.mark.parametrize("ne", [(1, 1, 1), (3, 1, 5), (7, 5, 3), (1, 9, 15), (16, 8, 8), (33, 29, 20)])
def test_step_matches_the_composed_step(ne):
    print(f"closure step {ne}", flush=True)
    dt = 0.002
    s = dg_amd.Solver(dg_amd.case_toml(order=1, basis="LegendreHex", flux="Roe", nelem=ne, lower=(-5., -4., -3.),
                                       upper=(5., 4., 3.), stepper="RK4", timestep=dt, ic="ExtrudedIsentropicVortex",
                                       ic_data=(1.0, 0.7, -0.4, 1.0, 3.0, 0.3, -0.2)))
    m = network()
    with s:
        s.init_state_from_fcn()
        U0 = s.get_state()
        u, r = hip.Buffer(U0.size), hip.Buffer(U0.size)
        E, largest = U0.shape[0], []

        def tendency(U):
            u.upload(U)
            s.get_residual(u.addr, r.addr)
            s.mult_inv_mass_matrix(dt, r.addr, r.addr)
            X = closure.features(s, u.addr.value if hasattr(u.addr, "value") else u.addr)
            hip.synchronize()
            C = m.forward(X, E).download((E, 8, 5))
            largest.append(np.max(np.abs(C)))
            return r.download(U.shape) + dt * C.astype(np.float64)

        k1 = tendency(U0)
        k2 = tendency(U0 + 0.5 * k1)
        k3 = tendency(U0 + 0.5 * k2)
        k4 = tendency(U0 + k3)
        ref = U0 + (k1 + 2.0 * k2 + 2.0 * k3 + k4) / 6.0
        closure.step(s, m, 1e30, 1)
        U1 = s.get_state()
        u.free()
        r.free()
    m.close()
    # the first stage sees the same features; later ones differ in their last
    # place, and an activation on a rounding boundary of bf16 (2^-8) can then
    # move an output: at most dt times a hundredth of the largest correction
    assert np.all(np.isfinite(U1)) and min(largest) > 0.0
    assert np.max(np.abs(U1 - ref)) <= 1e-13 * np.max(np.abs(ref)) + 0.01 * dt * max(largest)


@pytest.mark.parametrize("rows", [16384, 16385, 16511, 32769])
def test_forward_rows(rows):
    print(f"closure forward, {rows} rows", flush=True)
    rng = np.random.default_rng(3)
    X = rng.normal(0, 1, (rows, MO.NF)).astype(np.float32)
    m = network()
    Xd = hip.Buffer.from_array(X, np.float32)
    out = m.forward(Xd, rows).download((rows, MO.NO))
    for first, n in ((0, 200), (rows - 77, 77)):                   # the same rows in a small call
        part = hip.Buffer.from_array(X[first:first + n], np.float32)
        assert np.array_equal(m.forward(part, n).download((n, MO.NO)), out[first:first + n])
    m.close()
