"""The two passes where their workgroups end: element counts that fill the
last workgroup of both passes, leave one element in it, or one too few, at
every order in both precisions, above the sizes from which steps of both run in
two passes."""
import numpy as np
import pytest

from dg_amd import hip
from test_gpu_two_pass import composed, solver

pytestmark = pytest.mark.gpu

# elements per workgroup of the face and of the element pass, p = 1 .. 5, and
# the elements from which FP32 steps run in two passes (FP64 ones before)
EPB = [(7, 6), (5, 4), (4, 5), (3, 7), (3, 2)]
FROM = [7168, 5120, 5888, 14848, 8192]

CASES = []
for p in range(1, 6):
    f, g = EPB[p - 1]
    full = (FROM[p - 1] // (f * g) + 1) * f * g            # a multiple of both
    for k, n in enumerate((full, full + 1, full - 1)):
        ne = [1, 1, 1]
        ne[(p + k) % 3] = n
        CASES.append((p, tuple(ne), ("LegendreHex", "LagrangeHex")[(p + k) % 2],
                      ("Roe", "HLLC", "LaxFriedrichs")[(p + 2 * k) % 3]))


@pytest.mark.parametrize("order,ne,basis,flux", CASES)
@pytest.mark.parametrize("precision", [None, "FP32"])
def test_last_workgroups(order, ne, basis, flux, precision):
    print(f"two-pass edges p={order} {ne} {basis} {flux} {precision}", flush=True)
    eps = 2.0 ** -53 if precision is None else 2.0 ** -24
    s, dt = solver(order, ne, basis, flux, "RK4", precision)
    with s:
        U0 = s.get_state()
        u, ra, rb, st = hip.Buffer.from_array(U0), hip.Buffer(U0.size), hip.Buffer(U0.size), hip.Stream()
        s.get_residual(u.addr, ra.addr)                    # two passes; the fused kernel
        s.get_residual(u.addr, rb.addr, st.handle)
        hip.synchronize()
        a, b = ra.download(U0.shape), rb.download(U0.shape)
        for buf in (u, ra, rb):
            buf.free()
        s.take_time_step()
        U1 = s.get_state()
        ref = composed(s, U0, dt, "RK4")
    # the bounds of test_gpu_two_pass.py
    h = sorted((hi - lo) / n for lo, hi, n in zip((-5., -4., -3.), (5., 4., 3.), ne))
    size = 5. * np.max(np.abs(U0)) * h[1] * h[2]
    assert np.max(np.abs(b)) > 0.0
    assert np.max(np.abs(a - b)) <= 64 * eps * (np.max(np.abs(b)) + size)
    inc = np.max(np.abs(ref - U0))
    tol = 64 * eps * (2 * order + 1) ** 3 * inc + 4 * 2.0 ** -52 * np.max(np.abs(ref))
    assert inc > 0.0 and np.max(np.abs(U1 - ref)) <= tol
