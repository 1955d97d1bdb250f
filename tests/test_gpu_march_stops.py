"""A march that meets a dt that is not positive and finite stops there: as the
host loop of Compute_CFL, Compute_Tstep and LDDRK4 would, with the state, the
transport coefficients and the gradients as that dt found them, the clock of
the steps before it, the dt in the message, and without the time of the steps
that were asked for after it."""
import ctypes
import time

import numpy as np
import pytest

from fields import smooth_state

pytestmark = pytest.mark.gpu

st_amd = pytest.importorskip("st_amd")


def march(s, n, t, step):
    """st_march itself: (code, time, step, dts, message)."""
    tt, ss, d = np.array([t]), ctypes.c_int(step), np.full(n, -7.0)
    p = ctypes.POINTER(ctypes.c_double)
    rc = st_amd.lib().st_march(s.h, n, tt.ctypes.data_as(p), ctypes.byref(ss), d.ctypes.data_as(p))
    return rc, tt[0], ss.value, d, st_amd.lib().st_last_error(s.h).decode()


def same(a, b):
    return np.array_equal(a, b, equal_nan=True)


# an infinite coefficient makes its limit and so dt 0, a negative density a limit
# negative; fresh coefficients of the same state would give a valid dt again
@pytest.mark.parametrize("which", ["infinite coefficient", "negative density"])
@pytest.mark.parametrize("kw", [{}, {"rk_scheme": 2}, {"nonperiodic_x": 1}])
def test_recoverable_dt(which, kw):
    print("march stops", which, kw, flush=True)
    shape = (48, 32, 32)
    s = st_amd.Solver(*shape, Re=100.0, **kw)
    try:
        s.upload(smooth_state(*shape, seed=3, amp=0.1))
        s.march(2)
        Q, H, G = s.download(), s.hyper(), s.grad()
        if which == "negative density":
            Q[3, 4, 5, 3] = -0.25
            H[...] = 1e-3
        else:
            H[3, 4, 5, 1] = np.inf
        s.upload(Q)
        s.set_hyper(H)
        rc, t, step, d, said = march(s, 5, 0.5, 4)
        assert rc != 0 and (t, step) == (0.5, 4) and np.all(d == -7.0)
        dt = s.tstep(s.cfl()[1], 4)
        assert not dt > 0.0 and "dt %g at step 4" % dt in said
        assert same(s.download(), Q) and same(s.hyper(), H) and same(s.grad(), G)
    finally:
        s.close()


def test_later_step_of_a_chunk():
    shape = (16, 16, 16)
    kw = dict(Re=500.0, cfl_cal=1.0)                    # past the scheme's stability
    a, b = st_amd.Solver(*shape, **kw), st_amd.Solver(*shape, **kw)
    try:
        for s in (a, b):
            s.upload(smooth_state(*shape, seed=4, amp=0.5))
        t, n, dts = 0.25, 0, []
        while True:
            dt = b.tstep(b.cfl()[1], n)
            if not (dt > 0.0 and np.isfinite(dt)):
                break
            dts.append(dt)
            t, n = b.lddrk4(dt, t, n)
            assert n < 200
        assert n > 1
        rc, ta, na, d, said = march(a, 250, 0.25, 0)
        assert rc != 0 and (ta, na) == (t, n) and list(d[:n]) == dts and np.all(d[n:] == -7.0)
        assert "dt %g at step %d" % (dt, n) in said
        assert same(a.download(), b.download()) and same(a.hyper(), b.hyper()) and same(a.grad(), b.grad())
    finally:
        a.close()
        b.close()


def test_stops_soon():
    shape = (96, 96, 96)
    s = st_amd.Solver(*shape, Re=100.0)
    try:
        s.upload(smooth_state(*shape, seed=5, amp=0.3))
        s.march(4)                                      # warm
        t0 = time.perf_counter()
        s.march(16)
        ok = time.perf_counter() - t0
        Q = s.download()
        Q[..., 4] = np.nan
        s.upload(Q)
        t0 = time.perf_counter()
        rc = march(s, 256, 0.0, 4)[0]
        bad = time.perf_counter() - t0
        assert rc != 0 and bad < ok, (bad, ok)
    finally:
        s.close()
