"""The derivatives that a host program calls by themselves, point by point: the
response to an impulse keeps its digits down a line of 500 points, some 200
decades below its largest value, and a NaN or an infinity reaches its whole
line and no other.  The response is known in closed form: with the root r of
the operator's left side, the inverse of 1 + alpha (S + 1/S) on a ring of n
points is (r^d + r^(n-d)) / ((1 - r^n) sqrt(1 - 4 alpha^2))."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

st_amd = pytest.importorskip("st_amd")

OPS = {"d1": (1.0 / 3.0, {1: 14.0 / 18.0, 2: 1.0 / 36.0}, -1.0), "d2": (2.0 / 11.0, {1: 12.0 / 11.0, 2: 3.0 / 44.0}, 1.0)}


def response(op, n):
    """Row i: the operator (spacing 2 pi / n) at i points past a unit impulse."""
    al, w, sign = OPS[op]
    al = np.longdouble(al)
    root = np.sqrt(1 - 4 * al * al)
    r = (root - 1) / (2 * al)
    d = np.arange(n)
    g = (r ** d + r ** (n - d)) / ((1 - r ** n) * root)
    h = np.longdouble(2 * np.pi) / n
    out = np.zeros(n, np.longdouble)
    for m, a in w.items():                       # f(i + m) is the impulse at i = -m
        out += np.longdouble(a) * (sign * g[(d - m) % n] + g[(d + m) % n])
    if op == "d2":
        out -= 2 * sum(np.longdouble(a) for a in w.values()) * g
    return out / h ** (1 if op == "d1" else 2)


@pytest.mark.parametrize("n", [64, 80, 128, 224, 256, 320, 512])
def test_response_keeps_its_digits(n):
    for d in range(3):
        dims = [16, 16, 16]
        dims[d] = n
        print("tails", dims, d, flush=True)
        s = st_amd.Solver(*dims)
        axis = {0: 2, 1: 0, 2: 1}[d]
        at = [3, 5, 7]
        at[axis] = n // 2 + 3
        F = np.zeros(s.shape, order="F")
        F[tuple(at)] = 1.0
        line = [slice(k, k + 1) for k in at]
        line[axis] = slice(None)
        for narrow in (0, 1):
            s.set_pass_configs({"d1.%s" % "xyz"[d]: (narrow, 256), "d2.%s" % "xyz"[d]: (narrow, 256)})
            for op, got in (("d1", s.dfd(d, F)), ("d2", s.d2fd2(d, F))):
                ref = np.roll(response(op, n), at[axis])
                # in the middle opposite the impulse the two sides of D1 cancel
                far = np.abs((np.arange(n) - at[axis]) % n - n // 2) > 4
                # and so they do at the impulse, from the size of its neighbours
                size = np.abs(ref)
                size[at[axis]] = size.max()
                # each point: a chain of n multiplications by rounded powers of the root
                assert np.all(np.abs(got[tuple(line)].ravel() - ref)[far] <= 4 * n * 2.0 ** -53 * size[far]), (op, narrow)
                got[tuple(line)] = 0.0
                assert not got.any()
        s.close()


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("nonper", [0, 1])
@pytest.mark.parametrize("n", [64, 128, 256, 448, 512])
def test_not_finite_reaches_its_line(n, nonper, bad):
    for d in range(1 if nonper else 3):
        dims = [16, 16, 16]
        dims[d] = n
        s = st_amd.Solver(*dims, nonperiodic_x=nonper)
        axis = {0: 2, 1: 0, 2: 1}[d]
        at = [3, 5, 7]
        at[axis] = n - 20
        rng = np.random.default_rng(n)
        F = np.asfortranarray(rng.normal(size=s.shape))
        F[tuple(at)] = bad
        line = [slice(k, k + 1) for k in at]
        line[axis] = slice(None)
        for got in (s.dfd(d, F), s.d2fd2(d, F)):
            assert not np.isfinite(got[tuple(line)]).any(), (n, d)
            got[tuple(line)] = 0.0
            assert np.isfinite(got).all(), (n, d)
        s.close()
