"""dg_residual's two routes above the size of the two passes: on the handle's
stream the two passes, on the caller's own and under capture the fused
kernel, which uses no memory of the handle's.  A captured residual, replayed on
another stream beside the handle's own residuals, gives the fused kernel's
bits every time; in the FP32 form the routes give the same bits."""
import ctypes as C

import numpy as np
import pytest

from dg_amd import hip
from test_gpu_two_pass import solver

pytestmark = pytest.mark.gpu


def rt(name, *args):
    hip.check(getattr(hip.rt(), name)(*args), name)


@pytest.mark.parametrize("order,ne,precision", [(1, (17, 17, 16), None), (3, (14, 15, 14), None),
                                                (2, (18, 17, 17), "FP32")])
def test_captured_residual_is_the_fused_one(order, ne, precision):
    print(f"captured residual p={order} {ne} {precision}", flush=True)
    s, _ = solver(order, ne, "LegendreHex", "Roe", "RK4", precision)
    own, other = hip.Stream(), hip.Stream()
    with s:
        s.set_stream(own.handle)
        U = s.get_state()
        V = np.roll(U, 1, axis=0)
        u, v = hip.Buffer.from_array(U), hip.Buffer.from_array(V)
        r, rv, ref, refv = (hip.Buffer(U.size) for _ in range(4))
        s.get_residual(u.addr, ref.addr, other.handle)     # fused
        s.get_residual(v.addr, refv.addr)                  # two passes
        hip.synchronize()
        want, want_v = ref.download(), refv.download()
        graph, exe = C.c_void_p(), C.c_void_p()
        rt("hipStreamBeginCapture", own.h, 1)              # thread-local mode
        s.get_residual(u.addr, r.addr)                     # the handle's stream
        rt("hipStreamEndCapture", own.h, C.byref(graph))
        rt("hipGraphInstantiate", C.byref(exe), graph, None, None, C.c_size_t(0))
        zero = np.zeros(U.size)
        for k in range(8):
            r.upload(zero)
            rv.upload(zero)
            # the handle's residual of another state beside the replay
            s.get_residual(v.addr, rv.addr)
            rt("hipGraphLaunch", exe, other.h)
            s.get_residual(v.addr, rv.addr)
            hip.synchronize()
            assert np.array_equal(r.download(), want), k
            assert np.array_equal(rv.download(), want_v), k
            s.take_time_step()                             # and its steps in between
        rt("hipGraphExecDestroy", exe)
        rt("hipGraphDestroy", graph)
        s.set_stream(None)
        for b in (u, v, r, rv, ref, refv):
            b.free()
    own.destroy()
    other.destroy()


FP32 = [(1, (20, 19, 20)), (2, (18, 17, 17)), (3, (18, 17, 18)), (4, (25, 25, 24)), (5, (20, 19, 18))]


@pytest.mark.parametrize("order,ne", FP32)
@pytest.mark.parametrize("basis", ["LegendreHex", "LagrangeHex"])
@pytest.mark.parametrize("flux", ["Roe", "HLLC", "LaxFriedrichs"])
def test_fp32_routes_agree_to_the_bit(order, ne, basis, flux):
    print(f"FP32 residual routes p={order} {ne} {basis} {flux}", flush=True)
    s, _ = solver(order, ne, basis, flux, "RK4", "FP32")
    st = hip.Stream()
    with s:
        U = s.get_state()
        # the smooth state, then jumps at every face
        for W in (U, U * (1.0 + 0.05 * np.random.default_rng(5).standard_normal(U.shape))):
            s.set_state(W)
            u, a, b = hip.Buffer.from_array(W), hip.Buffer(W.size), hip.Buffer(W.size)
            s.get_residual(u.addr, a.addr)
            s.get_residual(u.addr, b.addr, st.handle)
            hip.synchronize()
            A, B = a.download(), b.download()
            for q in (u, a, b):
                q.free()
            assert np.max(np.abs(B)) > 0.0 and np.all(np.isfinite(B))
            assert np.array_equal(A, B)
    st.destroy()
