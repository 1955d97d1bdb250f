"""The artificial-transport coefficients after a whole step: the stages before
the last do not store them, so what a step leaves must be what the last stage
of the same step, run stage by stage, leaves (the same bits), for each RK
scheme, and so the next dt limit."""
import numpy as np
import pytest

import oracle as O
from fields import smooth_state

pytestmark = pytest.mark.gpu

st_amd = pytest.importorskip("st_amd")


@pytest.mark.parametrize("scheme", [0, 1, 2])
@pytest.mark.parametrize("shape,nonper", [((32, 32, 32), 0), ((48, 16, 32), 1)])
def test_step_leaves_the_last_stages_coefficients(shape, nonper, scheme):
    print("coefficients", shape, nonper, scheme, flush=True)
    kw = dict(Re=150.0, rk_scheme=scheme, nonperiodic_x=nonper)
    Q = smooth_state(*shape, seed=4, amp=1.2, mt=0.5)
    dt = 1.0e-3
    a, b = st_amd.Solver(*shape, **kw), st_amd.Solver(*shape, **kw)
    try:
        a.upload(Q)
        b.upload(Q)
        for step in range(2):
            a.lddrk4(dt)
            for loop in range(2):
                ra, rb = O.rk_coeffs(scheme, loop)
                for k in range(len(ra)):
                    b.rk_stage(ra[k], rb[k], dt, reset_qw=k == 0)
            H = a.hyper()
            assert np.abs(H).max() > 0 and np.array_equal(H, b.hyper()), step
            assert np.array_equal(a.download(), b.download()), step
            assert a.tstep(a.cfl()[1], 2) == b.tstep(b.cfl()[1], 2)
    finally:
        a.close()
        b.close()
