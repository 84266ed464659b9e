"""The trailing update of many tiles whose side 128 does not divide."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def update(dev, dtype):
    return dev.M.mi_dpotrf_step_update if dtype == np.float64 else dev.M.mi_spotrf_step_update


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("N,NB", [(2500, 64), (3200, 96), (3000, 160), (4000, 208), (3900, 320), (2600, 72),
                                  (2900, 80), (4100, 112)])
def test_many_tiles(dev, N, NB, dtype):
    """At least 512 blocks of 128.  A sum of K products onto C in any order is
    within (K + 1) u (|C| + |A| |B|^T) of the exact one; numpy adds its share."""
    print(f"update N={N} NB={NB} {dtype.__name__}", flush=True)
    MT = (N + NB - 1) // NB
    assert MT * (MT - 1) // 2 * ((NB + 127) // 128) ** 2 >= 512 and NB % 128
    T = np.random.default_rng(N).uniform(-2.0, 2.0, MT * (MT + 1) // 2 * NB * NB).astype(dtype)
    d = dev.upload(T)
    dev.check(update(dev, dtype)(dev.h, N, NB, d, 0, 1, MT), "update")
    got = dev.download(d, T.shape, dtype).astype(np.float64)
    dev.free(d)
    T = T.astype(np.float64)
    u = (2.0 ** -53 if dtype == np.float64 else 2.0 ** -24) + 2.0 ** -53

    def tile(X, m, k):
        i = k * MT - k * (k - 1) // 2 + (m - k)
        return X[i * NB * NB:(i + 1) * NB * NB].reshape((NB, NB), order="F")

    for k in range(1, MT):
        for m in range(k, MT):
            tm, tn = min(NB, N - m * NB), min(NB, N - k * NB)
            C, g, X, Y = tile(T, m, k), tile(got, m, k), tile(T, m, 0)[:tm], tile(T, k, 0)[:tn]
            low = np.tril(np.ones((tm, tn), bool)) if m == k else np.ones((tm, tn), bool)
            tol = (NB + 1) * u * (np.abs(C[:tm, :tn]) + np.abs(X) @ np.abs(Y).T)
            assert (np.abs(g[:tm, :tn] - (C[:tm, :tn] - X @ Y.T)) <= tol)[low].all(), (m, k)
            assert np.array_equal(g[:tm, :tn][~low], C[:tm, :tn][~low])
            assert np.array_equal(g[tm:], C[tm:])


def best_time(dev, N, NB, dtype):
    MT = (N + NB - 1) // NB
    n = MT * (MT + 1) // 2 * NB * NB * np.dtype(dtype).itemsize
    d = dev.alloc(n)
    dev.check(dev.M.mi_memset(dev.h, d, 0, n), "memset")
    times = []
    for _ in range(12):
        t = time.perf_counter()
        dev.check(update(dev, dtype)(dev.h, N, NB, d, 0, 1, MT), "update")
        times.append(time.perf_counter() - t)
    dev.free(d)
    return min(times)


def test_single_precision_takes_no_longer(dev):
    """Half the bytes and twice the matrix rate: an update of tiles of 64 in
    FP32 takes no longer than in FP64 (blocks of 128 took three times as long)."""
    f64, f32 = (best_time(dev, 8000, 64, t) for t in (np.float64, np.float32))
    print(f"FP64 {f64 * 1e6:.1f} us, FP32 {f32 * 1e6:.1f} us")
    assert f32 <= f64


def test_tiles_of_80_pad_to_96(dev):
    """Tiles of 64 have no padding.  Tiles of 80 padded to 96 take (96 / 80)^2
    times the work at a K longer by 80 / 64, 1.8 times the time; padded to 128
    they would take 3.2 times.  The bound is a quarter above the first."""
    t64, t80 = (best_time(dev, 8000, NB, np.float64) for NB in (64, 80))
    print(f"NB=64 {t64 * 1e6:.1f} us, NB=80 {t80 * 1e6:.1f} us")
    assert t80 <= 2.25 * t64
