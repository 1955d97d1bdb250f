"""D2 of a constant is 0, not a rounding of it divided by the spacing squared,
on lines of every length, direction and layout; and so are the second
derivatives that a right-hand side takes of a state at rest."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

st_amd = pytest.importorskip("st_amd")

LINES = (16, 32, 40, 48, 56, 64, 80, 96, 112, 128, 160, 192, 224, 256, 320, 384, 448, 512)


@pytest.mark.parametrize("n", LINES)
def test_constant(n):
    for d in range(3):
        dims = [16, 16, 16]
        dims[d] = n
        s = st_amd.Solver(*dims)
        for narrow in (0, 1):
            s.set_pass_configs({"d2.%s" % "xyz"[d]: (narrow, 256)})
            for c in (1.0, 27.78, 1.0 / 3.0, -0.1, 19.84, 7.1e-5):
                assert not s.d2fd2(d, np.full(s.shape, c, order="F")).any(), (n, d, narrow, c)
        s.close()


@pytest.mark.parametrize("shape", [(32, 48, 64), (128, 80, 56)])
def test_state_at_rest(shape):
    s = st_amd.Solver(*shape, Re=10.0)
    try:
        Q = np.zeros(s.shape + (5,), order="F")
        Q[..., 3], Q[..., 4] = 1.1, 17.3
        r = s.hyper_rhs(s.rhs(Q))
        assert not r.any()
    finally:
        s.close()
