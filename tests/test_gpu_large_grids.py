"""Grids just above the size from which passes stream and take the wide tiles
(STREAM_POINTS in csrc/st_kernels.h): line lengths of every kind in every
direction (5, 6 and 7 times a power of two beside the powers), the start-up
passes and one whole step (11 stages, with the fused passes between stages)
against the oracle.

Tolerances, max|gpu - cpu| / max|cpu| per field, those that the same
quantities have elsewhere: gradients 1e-13, start-up coefficients 1e-11
(times (n/256)^4 for lines n > 256), one step 1e-11 as at 256^3.  Where the
oracle's own spread under 1-ulp moves of Q is larger (the one-sided rows of a
non-periodic x), three times it for the coefficients, ten times it for a step
and its dt.
"""
import numpy as np
import pytest

import oracle as O
from fields import relerr, smooth_state

pytestmark = pytest.mark.gpu

st_amd = pytest.importorskip("st_amd")

STREAM_POINTS = 3 << 19


@pytest.mark.parametrize("shape,nonper", [
    ((128, 160, 80), 0), ((224, 64, 112), 0), ((64, 128, 192), 0), ((96, 112, 160), 0),
    ((512, 64, 48), 0), ((320, 48, 128), 1), ((192, 96, 96), 1)])
def test_startup_and_step_of_a_streaming_grid(shape, nonper):
    print("large grid", shape, "nonper", nonper, flush=True)
    assert np.prod(shape) >= STREAM_POINTS
    per = (2.0, 2 * np.pi, 2 * np.pi) if nonper else (2 * np.pi,) * 3
    kw = dict(Re=150.0, Pr=0.7, hyper_param=1, period=per)
    Q = smooth_state(*shape, seed=9, amp=1.1, mt=0.4)
    s = st_amd.Solver(*shape, nonperiodic_x=nonper, **kw)
    o = O.Oracle(*shape, nonper_x=nonper, **kw)
    try:
        Qp = np.asfortranarray(Q * (1 + np.random.default_rng(0).choice([-1, 1], size=Q.shape) * 2.2e-16))
        o2 = O.Oracle(*shape, nonper_x=nonper, **kw)
        o.compute_grad(Q)
        o2.compute_grad(Qp)
        Gc, Gp = o.grad()[..., :9], o2.grad()[..., :9]
        Hc, Hp = o.compute_hyper(Q).copy(), o2.compute_hyper(Qp).copy()
        Qc, _, _, dc = o.march(Q, 1)
        Qcp, _, _, dp = o2.march(Qp, 1)
        s.upload(Q)
        s.compute_grad()
        e, sp = relerr(s.grad()[..., :9], Gc).max(), relerr(Gp, Gc).max()
        print("  grad", e, "spread", sp, flush=True)
        assert e < max(1e-13, 3 * sp)
        e, sp = relerr(s.compute_hyper(), Hc).max(), relerr(Hp, Hc).max()
        print("  hyper", e, "spread", sp, flush=True)
        assert e < max(1e-11 * max(1.0, (max(shape) / 256.0) ** 4), 3 * sp)
        _, _, dg = s.march(1)
        e, sp = relerr(s.download(), Qc).max(), relerr(Qcp, Qc).max()
        print("  step", e, "spread", sp, "dt", dg[0], dc[0], dp[0], flush=True)
        assert abs(dg[0] - dc[0]) <= max(1e-12 * dc[0], 10 * abs(dp[0] - dc[0]))
        assert e < max(1e-11, 10 * sp)
    finally:
        s.close()
