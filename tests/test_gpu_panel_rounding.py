"""The solve of a panel's rows rounds once at the size of C.

The diagonal tile is the identity but for the last 16 columns' worth of rows
of each sub-column of 128, whose entries left of their diagonal block are
small integers times 2^-60 (FP64) or 2^-30 (FP32); the rows to solve hold
small integers in all other columns and arbitrary values in [1, 2) in those.
Then X = C in the other columns, and in the last ones X = C - s with s a sum
of integers below 2^13 times the same power of two, exact in any order: X is
the correctly rounded difference, bit for bit."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("NB,rows", [(32, 32), (93, 50), (100, 17), (128, 128), (137, 137), (160, 64), (256, 200)])
def test_rows_round_once(dev, NB, rows, dtype):
    print(f"panel rounding NB={NB} rows={rows} {dtype.__name__}", flush=True)
    N = NB + rows
    rng = np.random.default_rng(NB)
    ulp = 2.0 ** (-60 if dtype == np.float64 else -30)
    L, C = np.eye(NB), rng.integers(1, 9, (NB, NB)).astype(np.float64)
    last = []                                                   # (first column of the sub-column, of its last block)
    for c0 in range(0, NB, 128):
        w = min(128, NB - c0)
        l0 = c0 + (w - 1) // 16 * 16
        last.append((c0, l0, c0 + w))
        L[l0:c0 + w, c0:l0] = rng.integers(-8, 9, (c0 + w - l0, l0 - c0)) * ulp
        C[:, l0:c0 + w] = rng.uniform(1.0, 2.0, (NB, c0 + w - l0)).astype(dtype)
    T = np.concatenate([L.ravel(order="F"), C.ravel(order="F"), np.eye(NB).ravel(order="F")]).astype(dtype)
    d = dev.upload(T)
    M, info = dev.M, ctypes.c_int(-1)
    f = "d" if dtype == np.float64 else "s"
    dev.check(getattr(M, f"mi_{f}potrf_step_potrf")(dev.h, N, NB, d, 0, ctypes.byref(info)), "potrf")
    dev.check(getattr(M, f"mi_{f}potrf_step_trsm")(dev.h, N, NB, d, 0), "trsm")
    got = dev.download(d, T.shape, dtype)[NB * NB:2 * NB * NB].reshape((NB, NB), order="F")
    dev.free(d)
    assert info.value == 0
    exp = C.astype(dtype)
    for c0, l0, c1 in last:
        s = C[:, c0:l0] @ L[l0:c1, c0:l0].T                     # exact in double
        exp[:, l0:c1] = (C[:, l0:c1].astype(np.longdouble) - s).astype(dtype)
    assert np.array_equal(got[:rows], exp[:rows])
    assert np.array_equal(got[rows:], C[rows:].astype(dtype))
