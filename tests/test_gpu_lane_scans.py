"""The derivatives' line solves where their scans could lose a contribution:
impulses on lines of every lane layout (M and M/2 points per lane, rows of 8
to 64 lanes, one and several lines per wave), each at a place of its own
beside the ends of lanes, lane rows and lines, against the oracle's band solve.
The last lane row reaches around the line, so an impulse's response must
come back in at the other end, and none may leak into a neighbouring line."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

st_amd = pytest.importorskip("st_amd")

LINES = (16, 32, 40, 48, 56, 64, 80, 96, 112, 128, 160, 192, 224, 256, 320, 384, 448, 512)


def impulses(shape, axis):
    """One impulse per line, its place and size different from line to line."""
    n = shape[axis]
    F = np.zeros(shape, order="F")
    others = [k for k in range(3) if k != axis]
    i, j = np.meshgrid(*[np.arange(shape[k]) for k in others], indexing="ij")
    line = i + shape[others[0]] * j
    idx = [None] * 3
    idx[others[0]], idx[others[1]] = i, j
    idx[axis] = (line * 7 + line // 16) % n
    F[tuple(idx)] = 10.0 ** (line % 5 - 2)
    return F


@pytest.mark.parametrize("nonper", [0, 1])
@pytest.mark.parametrize("n", LINES)
def test_impulse_response(n, nonper):
    for d in range(1 if nonper else 3):
        dims = [16, 16, 16]
        dims[d] = n
        print("impulse", dims, d, nonper, flush=True)
        s = st_amd.Solver(*dims, nonperiodic_x=nonper)
        o = O.Oracle(*dims, nonper_x=nonper)
        axis = {0: 2, 1: 0, 2: 1}[d]
        F = impulses(s.shape, axis)
        ref1, ref2 = o.dfd(d, F), o.d2fd2(d, F)
        # per line: an impulse 10^4 times smaller than its neighbour's is still resolved
        for narrow in (0, 1):
            s.set_pass_configs({"d1.%s" % "xyz"[d]: (narrow, 256), "d2.%s" % "xyz"[d]: (narrow, 256)})
            for got, ref, tol in ((s.dfd(d, F), ref1, 1e-13), (s.d2fd2(d, F), ref2, 1e-12 if nonper else 1e-13)):
                err = np.abs(got - ref).max(axis=axis)
                size = np.abs(ref).max(axis=axis)
                assert np.all(err <= tol * size), (n, d, narrow, (err / size).max())
        s.close()
