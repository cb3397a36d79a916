"""Device memory of the two-pass stage's scratch: what fitted the device
without it still fits (the library takes the scratch back when an allocation
of its own fails), a handle takes it only where as much again as its arrays
stays free, and the steps after it is gone are those of the fused stage."""
import ctypes as C

import numpy as np
import pytest

import dg_amd
from dg_amd import hip

pytestmark = pytest.mark.gpu

BIG = (128, 128, 128)
E = 128 ** 3
ARRAYS = 4 * 40 * 8 * E          # four registers of 40 values at p = 1
SCRATCH = 3 * 4 * 5 * 8 * E      # the lifted fluxes of three faces: 1.0 GB
WORK = 6 * 8 * E
SLACK = 64 << 20                 # what the runtime allocates beside them, and rounding to its pages


def free_bytes():
    f, t = C.c_size_t(), C.c_size_t()
    hip.synchronize()
    hip.check(hip.rt().hipMemGetInfo(C.byref(f), C.byref(t)), "hipMemGetInfo")
    return f.value


class Filler:
    """device memory taken until `leave` bytes are free"""

    def __init__(self, leave):
        self.parts = []
        while free_bytes() > leave + (4 << 20):
            p = C.c_void_p()
            hip.check(hip.rt().hipMalloc(C.byref(p), min(8 << 30, free_bytes() - leave)), "hipMalloc (filler)")
            self.parts.append(p)

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        for p in self.parts:
            hip.rt().hipFree(p)


def solver(ne=BIG, order=1):
    dt = 0.02 / max(ne) / (2 * order + 1)
    s = dg_amd.Solver(dg_amd.case_toml(order=order, basis="LegendreHex", flux="Roe", nelem=ne, timestep=dt,
                                       ic="ExtrudedIsentropicVortex", ic_data=(1.0, 0.7, -0.4, 1.0, 3.0)))
    s.init_state_from_fcn()
    return s


def step_tol(U0, U1, order, n=1):
    """of steps whose stages ran in two passes and fused: the bound of
    test_gpu_two_pass.py"""
    inc = np.max(np.abs(U1 - U0))
    return n * (64 * 2.0 ** -53 * (2 * order + 1) ** 3 * inc + 4 * 2.0 ** -52 * np.max(np.abs(U1)))


def test_a_second_handle_takes_the_first_ones_scratch():
    f0 = free_bytes()
    a = solver()
    assert f0 - free_bytes() >= ARRAYS + WORK + SCRATCH - SLACK
    U0 = a.get_state()
    a.take_time_step()
    U1 = a.get_state()
    # room for the second handle's arrays once the first one's scratch is gone
    with Filler(ARRAYS + WORK - SCRATCH // 2):
        print("a second handle beside a filled device", flush=True)
        b = solver()
        a.set_state(U0)
        a.take_time_step()
        b.take_time_step()
        Ua, Ub = a.get_state(), b.get_state()
        a.close()
        b.close()
    assert np.array_equal(Ua, Ub)
    assert np.max(np.abs(Ua - U1)) <= step_tol(U0, U1, 1)


def test_a_handle_leaves_room_for_its_arrays_again():
    f0 = free_bytes()
    with solver() as s:                                     # (and loads the kernels)
        assert f0 - free_bytes() >= ARRAYS + WORK + SCRATCH - SLACK
    # scratch or not, by what stays free beside it: half of the arrays, or all
    for left, taken in ((ARRAYS // 2, 0), (ARRAYS + 4 * SLACK, SCRATCH)):
        with Filler(ARRAYS + WORK + SCRATCH + left):
            print(f"a handle that leaves {left} bytes free", flush=True)
            f0 = free_bytes()
            with solver() as s:
                used = f0 - free_bytes()
            assert abs(used - (ARRAYS + WORK + taken)) <= SLACK, (used, left)


def test_a_batch_goes_on_without_its_scratch():
    # cases that run the fused stage alone and the two passes as a group:
    # 48 of 2744 elements at p = 5, 0.57 GB of scratch
    order, ne, n = 5, (14, 14, 14), 48
    scratch = n * 2744 * 3 * 36 * 5 * 8
    cases = [solver(ne, order) for _ in range(n)]
    U0 = cases[0].get_state()
    f0 = free_bytes()
    with dg_amd.Batch(cases) as batch:
        assert f0 - free_bytes() >= scratch - SLACK
        batch.step(1)
        U1 = cases[0].get_state()
        with Filler(ARRAYS + WORK - scratch // 2):
            print("a handle beside a batch on a filled device", flush=True)
            with solver() as s:
                s.take_time_step()
        assert f0 - free_bytes() <= SLACK
        for k in (1, 8):                                    # the step captured again, then tuned
            for c in cases:
                c.set_state(U0)
            batch.step(k)
            with solver(ne, order) as ref:
                ref.take_time_step(0.0, k)
                R = ref.get_state()
            for c in (cases[0], cases[n // 2], cases[-1]):
                U = c.get_state()
                assert np.max(np.abs(U - R)) <= step_tol(U0, R, order, k)
            if k == 1:
                assert np.max(np.abs(U1 - R)) <= step_tol(U0, R, order)
    for c in cases:
        c.close()


def test_a_refused_handle_leaves_no_error_behind():
    with Filler(ARRAYS // 2):
        print("a handle that does not fit", flush=True)
        with pytest.raises(dg_amd.DGError) as ei:
            solver()
        assert ei.value.status == 2 and "out of memory" in str(ei.value)
        # the next call does not report it
        with solver((4, 4, 4)) as s:
            s.take_time_step()
            assert np.all(np.isfinite(s.get_state()))


def test_a_batch_uses_its_cases_scratch():
    # both hold scratch of their own: 126 and 63 MB, twice the slack together
    made = [(solver(ne), solver(ne)) for ne in ((64, 64, 64), (64, 32, 64), (3, 2, 1))]
    batch_s, solo_s = [m[0] for m in made], [m[1] for m in made]
    U0 = [s.get_state() for s in solo_s]
    f0 = free_bytes()
    with dg_amd.Batch(batch_s) as batch:
        assert f0 - free_bytes() <= SLACK
        for n in (1, 2, 7):                                 # replays of the captured step, then the tuned one
            print(f"a batch on its cases' scratch, {n} steps", flush=True)
            for sb, so, U in zip(batch_s, solo_s, U0):
                sb.set_state(U)
                so.set_state(U)
            batch_s[0].take_time_step()                     # its scratch serves a step of its own in between
            batch_s[0].set_state(U0[0])
            batch.step(n)
            for sb, so, U in zip(batch_s, solo_s, U0):
                so.take_time_step(0.0, n)
                R = so.get_state()
                assert np.max(np.abs(sb.get_state() - R)) <= step_tol(U, R, 1, n)
        # a case's scratch is taken back: the batch goes on without it
        with Filler(ARRAYS + WORK - (48 << 20)):
            with solver() as s:
                s.take_time_step()
        for sb, U in zip(batch_s, U0):
            sb.set_state(U)
        batch.step(7)
        for sb, so, U in zip(batch_s, solo_s, U0):
            R = so.get_state()
            assert np.max(np.abs(sb.get_state() - R)) <= step_tol(U, R, 1, 7)
    for s in batch_s + solo_s:
        s.close()
