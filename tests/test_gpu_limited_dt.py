"""Runs whose dt is set by the limits of the artificial transport, on boxes
coarse in x (the limits hold dx^2 against coefficients with dx^6 over the other
sides' fourth differences).  Grid-scale dilatation grows there, and dt, the
minimum of a limit over the points, magnifies what the state's rounding is by
three to five decades.  So the bound on each step's dt is the scheme's own: how
far the oracle's dt moves when its initial state is disturbed by the rounding
of the compact filter, whose solve divides the Nyquist mode by 1 - 2 alpha +
2 beta = 1.3e-3 (a rounding becomes 8.7e-14), of each of two implementations;
ten times the largest of four such moves, as each stage adds its own."""
import numpy as np
import pytest

import oracle as O
from fields import FILT_AL, FILT_BE

pytestmark = pytest.mark.gpu

st_amd = pytest.importorskip("st_amd")

NOISE = 2.0 * 2.0 ** -53 / (1.0 - 2.0 * FILT_AL + 2.0 * FILT_BE)


@pytest.mark.parametrize("shape,seed,rk", [((16, 32, 32), 2, 0), ((16, 32, 16), 1, 0), ((16, 48, 32), 1, 0),
                                           ((16, 32, 16), 3, 1)])
def test_dt_of_a_limited_run(shape, seed, rk):
    print("limited dt", shape, seed, rk, flush=True)
    kw = dict(Re=st_amd.re_for_taylor(40.0, 4.0, 1.0, 0.3), Pr=0.7, hyper_param=1, rk_scheme=rk)
    Q = np.asfortranarray(st_amd.ic_isotropic(*shape, k0=4.0, urms=1.0, mt=0.3, seed=seed))
    o = O.Oracle(*shape, **kw)
    want, cfl = [], []
    q, t, n = Q, 0.0, 0
    for _ in range(5):
        cfl.append(o.params.cfl_cal / o.cfl(q)[1])
        q, t, n, d = o.march(q, 1, t, n)
        want += d
    want, cfl = np.array(want), np.array(cfl)
    assert np.any(want < 0.99 * cfl)                    # the limits do set dt
    moved = []
    for k in range(4):
        P = Q * (1.0 + NOISE * np.random.default_rng(k).standard_normal(Q.shape))
        moved.append(np.abs(np.array(o.march(np.asfortranarray(P), 5)[3]) / want - 1.0))
    tol = 10.0 * np.max(moved, axis=0) + 1e-12
    s = st_amd.Solver(*shape, **kw)
    try:
        s.upload(Q)
        dts = s.march(5)[2]
        off = np.abs(np.array(dts) / want - 1.0)
        assert np.all(off <= tol), (off, tol)
    finally:
        s.close()
