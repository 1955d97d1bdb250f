"""The march's dt and clock, formed on the device: the same bits as
Compute_CFL, Compute_Tstep and LDDRK4 called one by one from the host, for
one and many reduction blocks, with and without the limits of the artificial
transport, over more steps than one host synchronisation covers; and a step
whose dt is not positive and finite fails without touching the state."""
import numpy as np
import pytest

from fields import smooth_state

pytestmark = pytest.mark.gpu

st_amd = pytest.importorskip("st_amd")


@pytest.mark.parametrize("shape,kw", [((16, 16, 16), {}), ((64, 64, 64), {}), ((32, 32, 32), {"hyper_param": 0, "rk_scheme": 2}),
                                      ((48, 16, 32), {"nonperiodic_x": 1}), ((128, 64, 80), {"rk_scheme": 1})])
def test_march_is_the_host_loop(shape, kw):
    print("march clock", shape, kw, flush=True)
    Q = smooth_state(*shape, seed=7, amp=1.3, mt=0.5)
    a, b = st_amd.Solver(*shape, Re=200.0, **kw), st_amd.Solver(*shape, Re=200.0, **kw)
    try:
        a.upload(Q)
        b.upload(Q)
        b.compute_hyper()
        a.compute_hyper()
        ta, sa, dts = a.march(5, time=0.25, step=0)
        tb, sb, host = 0.25, 0, []
        for _ in range(5):
            host.append(b.tstep(b.cfl()[1], sb))
            tb, sb = b.lddrk4(host[-1], tb, sb)
        assert list(dts) == host and ta == tb and sa == sb == 5
        assert np.array_equal(a.download(), b.download())
    finally:
        a.close()
        b.close()


def test_march_across_chunks():
    shape = (16, 16, 16)
    Q = smooth_state(*shape, seed=8)
    a, b = st_amd.Solver(*shape, Re=100.0), st_amd.Solver(*shape, Re=100.0)
    try:
        a.upload(Q)
        b.upload(Q)
        t, s, dts = a.march(600)
        u, r = 0.0, 0
        parts = []
        for n in (1, 255, 1, 300, 43):
            u, r, d = b.march(n, time=u, step=r)
            parts += list(d)
        assert (t, s) == (u, r) and s == 600 and list(dts) == parts
        assert np.array_equal(a.download(), b.download())
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("hyper", [0, 1])
def test_invalid_dt_leaves_the_state(hyper):
    shape = (16, 16, 16)
    Q = smooth_state(*shape, seed=9)
    Q[..., 4] = np.nan                       # no point has a sound speed
    s = st_amd.Solver(*shape, Re=100.0, hyper_param=hyper)
    try:
        s.upload(Q)
        with pytest.raises(st_amd.StError, match="dt"):
            s.march(3, time=1.0, step=4)
        assert np.array_equal(s.download(), Q, equal_nan=True)
    finally:
        s.close()
