"""Host arrays that the caller has pinned: byte for byte as pageable ones, and
at the rate of a plain copy between pinned and device memory."""
import ctypes
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
st_amd = pytest.importorskip("st_amd")


def _best(f, n=15):
    t = []
    for _ in range(n):
        t0 = time.perf_counter()
        f()
        t.append(time.perf_counter() - t0)
    return min(t)


@pytest.mark.parametrize("shape", [(32, 32, 32), (64, 64, 64), (112, 80, 96)])
def test_pinned_states(shape):
    print("pinned", shape, flush=True)
    s = st_amd.Solver(*shape, Re=100.0)
    L, p = st_amd.lib(), ctypes.POINTER(ctypes.c_double)
    try:
        n = 5 * int(np.prod(shape))
        a, b = (torch.empty(n, dtype=torch.float64, pin_memory=True) for _ in range(2))
        d = torch.empty(n, dtype=torch.float64, device="cuda")
        a.copy_(torch.randn(n, dtype=torch.float64, generator=torch.Generator().manual_seed(1)))
        pa, pb = (ctypes.cast(t.data_ptr(), p) for t in (a, b))

        def up():
            assert L.st_state_upload(s.h, pa) == 0

        def down():
            assert L.st_state_download(s.h, pb) == 0

        def plain(dst, src):
            dst.copy_(src, non_blocking=True)
            torch.cuda.synchronize()

        up()
        down()
        assert torch.equal(a, b)
        assert np.array_equal(s.download().ravel(order="F"), a.numpy())
        if n * 8 >= 8 << 20:                 # where the rate and not the call counts
            assert _best(up) < 1.25 * _best(lambda: plain(d, a)) + 2e-5
            assert _best(down) < 1.25 * _best(lambda: plain(b, d)) + 2e-5
    finally:
        s.close()
