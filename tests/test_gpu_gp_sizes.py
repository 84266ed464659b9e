"""Tile sizes of the Gaussian-process calls: what is refused is refused before
anything is written."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("NB", [32, 544, 576, 608, 640, 672, 928, 960, 40, 992])
def test_tile_sizes(dev, NB, dtype):
    """Multiples of 32 up to 960 that the factorization takes: in FP64 above 560
    only multiples of 64.  K = 4 I: nll = N log 2 + 1/8 y^T y + N/2 log 2 pi."""
    print(f"gp NB={NB} {dtype.__name__}", flush=True)
    N = NB + 3
    MT = 2
    K = (4.0 * np.eye(N)).astype(dtype)
    y = np.full(N, 2.0, dtype)
    T = np.full(MT * (MT + 1) // 2 * NB * NB, 7.0, dtype)
    dK, dy, dT, do = dev.upload(K), dev.upload(y), dev.upload(T), dev.upload(np.full(2, 7.0))
    info = ctypes.c_int(-1)
    fn = dev.M.mi_dgp_nll if dtype == np.float64 else dev.M.mi_sgp_nll
    rc = fn(dev.h, N, NB, dK, N, dT, dy, do, ctypes.byref(info))
    gy, gT, go = dev.download(dy, y.shape, dtype), dev.download(dT, T.shape, dtype), dev.download(do, (2,))
    for p in (dK, dy, dT, do):
        dev.free(p)
    if NB % 32 or NB > 960:
        assert rc == -2
    elif dtype == np.float64 and NB > 560 and NB % 64:
        assert rc == -4
    else:
        assert rc == 0 and info.value == 0
        assert np.array_equal(gy, y / 2)
        assert abs(go[0] - N * np.log(2.0)) <= 1e-12 * N and abs(go[1] - N) <= 1e-12 * N
        return
    assert np.array_equal(gy, y) and np.array_equal(gT, T) and np.array_equal(go, [7.0, 7.0])
