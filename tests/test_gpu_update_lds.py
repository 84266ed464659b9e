"""The trailing update through LDS in each of its block sizes: 128 x 128
(launches of at least 512 such blocks), 64 x 64, and 32 x 32 (at most 256
blocks of 64), ragged last tiles, NaN in every row past the matrix.

A sum of K products onto C in any order is within (K + 1) u (|C| + |A| |B|^T)
of the exact one, element by element; numpy's FP64 reference adds its own
share."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("N,NB,block", [(600, 160, 32), (250, 64, 32), (1500, 128, 64), (1800, 192, 64), (1700, 320, 64),
                                        (5000, 512, 128), (4500, 384, 128)])
def test_update_blocks(dev, N, NB, block, dtype):
    print(f"update N={N} NB={NB} blocks of {block} {dtype.__name__}", flush=True)
    MT = (N + NB - 1) // NB
    count = lambda b: MT * (MT - 1) // 2 * ((NB + b - 1) // b) ** 2
    assert block == (128 if count(128) >= 512 else 32 if count(64) <= 256 else 64)
    rng = np.random.default_rng(N)
    T = rng.uniform(-2.0, 2.0, MT * (MT + 1) // 2 * NB * NB).astype(dtype)

    def tile(X, m, k):
        i = k * MT - k * (k - 1) // 2 + (m - k)
        return X[i * NB * NB:(i + 1) * NB * NB].reshape((NB, NB), order="F")

    last = N - (MT - 1) * NB
    for k in range(MT):
        tile(T, MT - 1, k)[last:] = np.nan
    tile(T, MT - 1, MT - 1)[:, last:] = np.nan
    d = dev.upload(T)
    fn = dev.M.mi_dpotrf_step_update if dtype == np.float64 else dev.M.mi_spotrf_step_update
    dev.check(fn(dev.h, N, NB, d, 0, 1, MT), "update")
    got = dev.download(d, T.shape, dtype)
    dev.free(d)
    u = (2.0 ** -53 if dtype == np.float64 else 2.0 ** -24) + 2.0 ** -53
    wide = lambda x: x.astype(np.float64)
    for k in range(1, MT):
        for m in range(k, MT):
            tm, tn = min(NB, N - m * NB), min(NB, N - k * NB)
            C, g = tile(T, m, k), tile(got, m, k)
            X, Y = wide(tile(T, m, 0)[:tm]), wide(tile(T, k, 0)[:tn])
            exp = wide(C[:tm, :tn]) - X @ Y.T
            tol = (NB + 1) * u * (np.abs(wide(C[:tm, :tn])) + np.abs(X) @ np.abs(Y).T)
            low = np.tril(np.ones((tm, tn), bool)) if m == k else np.ones((tm, tn), bool)
            assert (np.abs(wide(g[:tm, :tn]) - exp) <= tol)[low].all(), (m, k)
            assert np.array_equal(g[:tm, :tn][~low], C[:tm, :tn][~low])
            assert np.array_equal(g[tm:], C[tm:], equal_nan=True)
