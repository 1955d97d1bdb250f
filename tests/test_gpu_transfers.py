"""Host transfers at the sizes where their pieces change: below the staged
path, several fields in one piece, a field of exactly one piece, of one piece
and a remainder; whole states and slots of a batch, byte for byte."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

st_amd = pytest.importorskip("st_amd")

# (nx, ny, nz): a field is 32 KiB, 256 KiB (five in one piece), 960 KiB (two a
# piece, one left), 2 MiB, 2.2 MiB, 6.6 MiB
SHAPES = [(16, 16, 16), (32, 32, 32), (64, 48, 40), (64, 64, 64), (80, 64, 56), (112, 80, 96)]


def _state(shape, seed):
    nx, ny, nz = shape
    Q = np.asfortranarray(np.random.default_rng(seed).normal(scale=0.1, size=(ny, nz, nx, 5)))
    Q[..., 3] += 1.0
    Q[..., 4] += 9.0
    return Q


@pytest.mark.parametrize("shape", SHAPES)
def test_states_and_slots_round_trip(shape):
    print("transfers", shape, flush=True)
    b = st_amd.Batch(*shape, 3, Re=100.0)
    try:
        Qs = [_state(shape, k) for k in range(3)]
        for k, Q in enumerate(Qs):
            b.load(k, Q, 100.0, 1)
        for k, Q in enumerate(Qs):
            assert np.array_equal(b.store(k), Q), k
        b.upload(Qs[2])                                  # slot 0
        assert np.array_equal(b.download(), Qs[2])
        for k in (1, 2):
            assert np.array_equal(b.store(k), Qs[k]), k
        H = _state(shape, 9)[..., :3].copy(order="F")
        b.set_hyper(H)
        assert np.array_equal(b.hyper(), H)
    finally:
        b.close()
