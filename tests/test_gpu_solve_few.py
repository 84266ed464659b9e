"""Triangular solves with few right-hand sides (the wavefront on the VALU up
to 4, on the matrix cores from 5) at the edges of its 128-row blocks: one
element, ragged last blocks, tiles that blocks straddle, and NaN everywhere
that no entry of L lies.

Substitution by blocks of inverses errs, row by row, by at most about (N +
256) u |L^-1| |L| |x| (a sum of N products and two products of 128 terms);
the factor |L^-1| |L| is taken from the matrix."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("N,NB", [(1, 32), (31, 32), (127, 64), (128, 128), (129, 96), (257, 160), (385, 32), (641, 224),
                                  (1023, 256), (1500, 960)])
def test_few_right_hand_sides(dev, po, N, NB, dtype):
    rng = np.random.default_rng(N)
    B = rng.standard_normal((N, N))
    L = np.linalg.cholesky(B @ B.T / N + np.eye(N)).astype(dtype).astype(np.float64)
    Li = np.linalg.inv(L)
    T = po.full_to_symtiles(np.where(np.tri(N, dtype=bool), L, np.nan), NB)
    T[T == 0.0] = np.nan                                  # padding past N
    d = dev.upload(T.astype(dtype))
    fn = dev.M.mi_dtrsm_LL if dtype == np.float64 else dev.M.mi_strsm_LL
    try:
        for nrhs in (1, 2, 3, 4, 5):
            ldb = N + 3
            b = rng.standard_normal((nrhs, ldb)).astype(dtype)
            for trans in (111, 112):
                x = np.linalg.solve(L if trans == 111 else L.T, b[:, :N].astype(np.float64).T).T
                skeel = (np.abs(Li) @ np.abs(L) if trans == 111 else np.abs(Li.T) @ np.abs(L.T)).sum(axis=1).max()
                db = dev.upload(b)
                try:
                    dev.check(fn(dev.h, trans, 131, 1.0, N, NB, d, nrhs, db, ldb), "trsm")
                    got = dev.download(db, b.shape, dtype)
                finally:
                    dev.free(db)
                tol = (N + 256) * np.finfo(dtype).eps * skeel * np.abs(x).max()
                assert np.abs(got[:, :N] - x).max() <= tol, (nrhs, trans)
                assert np.array_equal(got[:, N:], b[:, N:])
    finally:
        dev.free(d)
