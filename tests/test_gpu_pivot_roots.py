"""The diagonal of a factor is the rounded root of its pivots.

Diagonal matrices: the pivots are the entries themselves.  The last step of
the root multiplies a residual below 2 ulp by a reciprocal good to 2^-20, so
the result is within (1/2 + 2^-18) ulp of the exact root (numpy's in long
double, itself within 2^-11 ulp)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(L, a):
    exact = np.sqrt(a.astype(np.longdouble))
    ulp = np.spacing(exact.astype(a.dtype)).astype(np.longdouble)
    assert (np.abs(L - exact) <= (0.5 + 2.0 ** -18 + 2.0 ** -11) * ulp).all()


def values(n, seed, dtype):
    rng = np.random.default_rng(seed)
    f = np.finfo(dtype)
    a = rng.uniform(1.0, 2.0, n) * 2.0 ** rng.integers(-40, 41, n)
    a[::7] = rng.uniform(1.0, 1.9, len(a[::7])) * 2.0 ** rng.integers(f.minexp, f.maxexp, len(a[::7])).astype(float)
    a[n // 2] = f.max
    a[n // 3] = f.tiny / 2 ** 10                               # a denormal: root and division
    return a.astype(dtype)


types = pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])


@types
@pytest.mark.parametrize("N,NB", [(16, 16), (93, 93), (300, 93), (400, 128), (513, 256)])
def test_roots_of_tiles(dev, po, N, NB, dtype):
    print(f"roots N={N} NB={NB} {dtype.__name__}", flush=True)
    a = values(N, N, dtype)
    T = po.full_to_symtiles(np.diag(a.astype(np.float64)), NB).astype(dtype)
    d = dev.upload(T)
    info = ctypes.c_int(-1)
    fn = dev.M.mi_dpotrf_tiles if dtype == np.float64 else dev.M.mi_spotrf_tiles
    dev.check(fn(dev.h, N, NB, d, ctypes.byref(info)), "potrf")
    got = dev.download(d, T.shape, dtype)
    dev.free(d)
    assert info.value == 0
    L = np.tril(po.symtiles_to_full(got.astype(np.float64), N, NB))
    check(L.diagonal(), a)
    assert not np.tril(L, -1).any()


@types
@pytest.mark.parametrize("n,count", [(3, 200), (17, 60), (64, 9), (100, 9), (128, 9), (300, 3)])
def test_roots_of_a_batch(dev, n, count, dtype):
    print(f"roots of {count} matrices of {n} {dtype.__name__}", flush=True)
    a = values(n * count, n, dtype).reshape(count, n)
    A = np.zeros((count, n, n), dtype)
    A[:, np.arange(n), np.arange(n)] = a
    p = ctypes.c_void_p()
    dev.check(dev.M.mi_batch_create(dev.h, count, (ctypes.c_int * count)(*[n] * count), ctypes.byref(p)), "create")
    d = dev.upload(A.ravel())
    try:
        fn = dev.M.mi_dposv_batched if dtype == np.float64 else dev.M.mi_sposv_batched
        dev.check(fn(p, d, None, 0), "posv_batched")
        got = dev.download(d, (count * n * n,), dtype).reshape(count, n, n)
    finally:
        dev.M.mi_batch_destroy(p)
        dev.free(d)
    check(got[:, np.arange(n), np.arange(n)], a)
