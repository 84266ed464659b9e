"""The trailing update of tiles that the LDS form does not take (odd sizes, K
not a multiple of 16) rounds once at the size of C.

u is the unit roundoff.  The K products add up from zero, within
(K + 1) u |A| |B|^T of their exact sum in any order, and the one subtraction
from C adds u |result|.  With |A|, |B| <= 2^-10 and 1 <= C < 2 the first part
is below u / 3 up to K = 520, while a sum that starts at C rounds at C's size
in every step.  The exact result is numpy's long double (FP64) or double
(FP32), whose own error is at most (K + 2) 2^-11 u."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("N,NB", [(30, 9), (200, 40), (300, 93), (300, 100), (290, 136), (500, 367), (700, 520)])
def test_one_rounding_at_c(dev, N, NB, dtype):
    print(f"rounding N={N} NB={NB} {dtype.__name__}", flush=True)
    wide = np.longdouble if dtype == np.float64 else np.float64
    u = 2.0 ** -53 if dtype == np.float64 else 2.0 ** -24
    MT = (N + NB - 1) // NB
    rng = np.random.default_rng(N)
    n = MT * (MT + 1) // 2 * NB * NB
    T = rng.uniform(1.0, 2.0, n)
    T[:MT * NB * NB] = rng.uniform(-2.0 ** -10, 2.0 ** -10, MT * NB * NB)       # tile column 0: A and B
    T = T.astype(dtype)
    d = dev.upload(T)
    fn = dev.M.mi_dpotrf_step_update if dtype == np.float64 else dev.M.mi_spotrf_step_update
    dev.check(fn(dev.h, N, NB, d, 0, 1, MT), "update")
    got = dev.download(d, T.shape, dtype).astype(wide)
    dev.free(d)
    T = T.astype(wide)

    def tile(X, m, k):
        i = k * MT - k * (k - 1) // 2 + (m - k)
        return X[i * NB * NB:(i + 1) * NB * NB].reshape((NB, NB), order="F")

    for k in range(1, MT):
        for m in range(k, MT):
            tm, tn = min(NB, N - m * NB), min(NB, N - k * NB)
            X, Y = tile(T, m, 0)[:tm], tile(T, k, 0)[:tn]
            exp = tile(T, m, k)[:tm, :tn] - X @ Y.T
            tol = u * np.abs(exp) + (NB + 1) * u * (np.abs(X) @ np.abs(Y).T) + (NB + 2) * 2.0 ** -11 * u
            err = np.abs(tile(got, m, k)[:tm, :tn] - exp)
            if m == k:
                err = np.tril(err)
            assert (err <= tol).all(), (m, k, float((err / tol).max()))


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("N,NB", [(30, 9), (200, 40), (300, 93), (700, 367)])
def test_infinity_in_the_last_column(dev, N, NB, dtype):
    """K is padded to whole stages by repeating its last column; an infinity
    there still gives infinities, not 0 * inf."""
    print(f"inf N={N} NB={NB} {dtype.__name__}", flush=True)
    MT = (N + NB - 1) // NB
    rng = np.random.default_rng(N)
    T = rng.uniform(1.0, 2.0, MT * (MT + 1) // 2 * NB * NB).astype(dtype)

    def tile(X, m, k):
        i = k * MT - k * (k - 1) // 2 + (m - k)
        return X[i * NB * NB:(i + 1) * NB * NB].reshape((NB, NB), order="F")

    for m in range(1, MT):
        tile(T, m, 0)[1, NB - 1] = np.inf
    d = dev.upload(T)
    fn = dev.M.mi_dpotrf_step_update if dtype == np.float64 else dev.M.mi_spotrf_step_update
    dev.check(fn(dev.h, N, NB, d, 0, 1, MT), "update")
    got = dev.download(d, T.shape, dtype)
    dev.free(d)
    for k in range(1, MT):
        for m in range(k, MT):
            tm, tn = min(NB, N - m * NB), min(NB, N - k * NB)
            low = np.tril(np.ones((tm, tn), bool)) if m == k else np.ones((tm, tn), bool)
            g = tile(got, m, k)[:tm, :tn]
            inf = np.zeros((tm, tn), bool)
            inf[1, :] = inf[:, 1] = True
            assert (g[low & inf] == -np.inf).all()
            assert np.isfinite(g[low & ~inf]).all()
