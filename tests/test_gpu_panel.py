"""The panel kernels of the tile Cholesky (sub-columns of 128 columns in
16 x 16 blocks) and the update kernel that streams its operands into LDS, at
the edges of their blocks, against the FP64 oracle and numpy.

Bounds: the factor of a diagonally dominant matrix is within a few n eps of
the exact one; 1e-12 of the largest entry in FP64 (as the other factor
tests) and 64 eps32 in FP32.  A sum of K products onto C in any order is
within (K + 1) eps (|C| + |A| |B|^T) of the exact one, element by element;
numpy's FP64 reference adds its own share."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS32 = 2.0 ** -24


def factor(dev, A, NB, dtype, rec=None):
    """Factor the dense A as tiles of NB; returns (lower factor, info)."""
    import pyoracle as po
    N = A.shape[0]
    T = po.full_to_symtiles(A, NB).astype(dtype)
    d = dev.upload(T)
    info = ctypes.c_int(-1)
    try:
        if rec:
            dev.check(dev.M.mi_dpotrf_tiles_rec(dev.h, N, NB, d, rec, ctypes.byref(info)), "potrf_rec")
        else:
            fn = dev.M.mi_dpotrf_tiles if dtype == np.float64 else dev.M.mi_spotrf_tiles
            dev.check(fn(dev.h, N, NB, d, ctypes.byref(info)), "potrf")
        got = dev.download(d, T.shape, dtype)
    finally:
        dev.free(d)
    return np.tril(po.symtiles_to_full(got.astype(np.float64), N, NB)), info.value


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("N,NB", [(1, 1), (1, 8), (15, 16), (16, 16), (17, 17), (31, 200), (127, 128), (128, 128),
                                  (129, 129), (143, 144), (250, 111), (257, 256), (300, 137), (385, 384), (401, 200),
                                  (513, 130), (777, 259)])
def test_panel_edges(dev, po, N, NB, dtype):
    print(f"panel N={N} NB={NB} {dtype.__name__}", flush=True)
    A = po.dplgsy_full(N, float(N), 3872).astype(dtype).astype(np.float64)
    L, info = factor(dev, A, NB, dtype)
    assert info == 0
    ref = np.linalg.cholesky(A)
    assert np.abs(L - ref).max() <= (1e-12 if dtype == np.float64 else 64 * EPS32) * np.abs(ref).max()


@pytest.mark.parametrize("hmb", [32, 64, 96, 128, 160])
def test_sub_column_widths(dev, po, hmb):
    N, NB = 500, 224
    A = po.dplgsy_full(N, float(N), 3872)
    L, info = factor(dev, A, NB, np.float64, rec=hmb)
    assert info == 0
    ref = np.linalg.cholesky(A)
    assert np.abs(L - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("scale", [2.0 ** -1000, 2.0 ** -1060, 2.0 ** 1000])
def test_pivots_near_the_ends_of_the_range(dev, po, scale):
    """The factor of s A is sqrt(s) times that of A.  Where entries and
    products are denormal every one of the at most N updates of an entry
    rounds to a multiple of 2^-1074, which the division by the pivot's root
    (at least its smallest diagonal entry) carries into L."""
    N, NB = 150, 150
    A = po.dplgsy_full(N, float(N), 3872)
    S = A * scale
    L, info = factor(dev, S, NB, np.float64)
    assert info == 0
    ref = np.linalg.cholesky(S / scale) * np.sqrt(scale)
    denormal = N * 2.0 ** -1074 / ref.diagonal().min()
    assert np.abs(L - ref).max() <= 1e-12 * np.abs(ref).max() + denormal


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("value", [0.0, -1.0, np.nan])
@pytest.mark.parametrize("bad", [0, 15, 16, 127, 128, 200, 299])
def test_bad_pivot(dev, po, bad, value, dtype):
    N, NB = 300, 300
    A = po.dplgsy_full(N, float(N), 3872)
    A[bad, bad] = value
    _, info = factor(dev, A, NB, dtype)
    assert info == bad + 1


def test_infinite_pivot_is_not_a_failure(dev, po):
    """As sqrt and division give it: L(j, j) = inf and zeros below it."""
    N, NB, j = 100, 100, 20
    A = po.dplgsy_full(N, float(N), 3872)
    A[j, j] = np.inf
    L, info = factor(dev, A, NB, np.float64)
    assert info == 0
    assert np.isinf(L[j, j]) and not L[j + 1:, j].any()
    keep = [i for i in range(N) if i != j]
    ref = np.linalg.cholesky(A[np.ix_(keep, keep)])
    assert np.abs(L[np.ix_(keep, keep)] - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("shift", [0, 1], ids=["aligned", "unaligned"])
@pytest.mark.parametrize("N,NB", [(300, 72), (500, 136), (1000, 200), (700, 176), (1100, 520), (2300, 100),
                                  (5300, 600)])
def test_update_shapes(dev, po, N, NB, shift, dtype):
    """K a multiple of 8 but not of 16, tiles that are no multiple of the
    block, ragged last tiles, and a tile image that starts off a 16-byte
    boundary (operands then go through registers); the last case runs the
    128 x 128 blocks."""
    print(f"update N={N} NB={NB} shift={shift} {dtype.__name__}", flush=True)
    MT = (N + NB - 1) // NB
    rng = np.random.default_rng(N)
    n = MT * (MT + 1) // 2 * NB * NB
    T = rng.uniform(-2.0, 2.0, n).astype(dtype)
    buf = np.concatenate([np.zeros(shift, dtype), T])
    d = dev.upload(buf)
    p = d + shift * buf.itemsize
    fn = dev.M.mi_dpotrf_step_update if dtype == np.float64 else dev.M.mi_spotrf_step_update
    dev.check(fn(dev.h, N, NB, p, 0, 1, MT), "update")
    got = dev.download(d, buf.shape, dtype)[shift:].astype(np.float64)
    dev.free(d)
    T = T.astype(np.float64)
    eps = (NB + 1) * ((2.0 ** -53 if dtype == np.float64 else EPS32) + 2.0 ** -53)

    def tile(X, m, k):
        i = k * MT - k * (k - 1) // 2 + (m - k)
        return X[i * NB * NB:(i + 1) * NB * NB].reshape((NB, NB), order="F")

    for k in range(1, MT):
        for m in range(k, MT):
            tm, tn = min(NB, N - m * NB), min(NB, N - k * NB)
            C, g = tile(T, m, k), tile(got, m, k)
            X, Y = tile(T, m, 0)[:tm], tile(T, k, 0)[:tn]
            exp = C[:tm, :tn] - X @ Y.T
            tol = eps * (np.abs(C[:tm, :tn]) + np.abs(X) @ np.abs(Y).T)
            low = np.tril(np.ones((tm, tn), bool)) if m == k else np.ones((tm, tn), bool)
            assert (np.abs(g[:tm, :tn] - exp) <= tol)[low].all()
            assert np.array_equal(g[:tm, :tn][~low], C[:tm, :tn][~low])
            assert np.array_equal(g[tm:], C[tm:])


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("unit", [False, True])
@pytest.mark.parametrize("trans", [111, 112])
@pytest.mark.parametrize("N,NB", [(1, 32), (15, 32), (17, 32), (127, 128), (129, 96), (145, 160), (257, 64),
                                  (400, 160), (529, 512)])
def test_wavefront_inverses_at_block_edges(dev, po, N, NB, trans, unit, dtype):
    """The 128-row inverses and link matrices of the wavefront solve, ragged
    in every way; the strict upper triangles and padding hold NaN.  With
    |off-diagonal| <= 1 / N and a diagonal in [1, 2] the inverse's entries
    stay below 2, so x is within a few N eps of the exact one."""
    print(f"wave N={N} NB={NB} {trans} {unit} {dtype.__name__}", flush=True)
    rng = np.random.default_rng(N + NB)
    A = rng.uniform(-1.0, 1.0, (N, N)) / N
    A[np.diag_indices(N)] = 1.0 + rng.uniform(0.0, 1.0, N)
    L = np.tril(A).astype(dtype).astype(np.float64)
    T = po.full_to_symtiles(L, NB).astype(dtype)
    MT = (N + NB - 1) // NB
    for n in range(MT):
        for m in range(n, MT):
            i = n * MT - n * (n - 1) // 2 + (m - n)
            t = T[i * NB * NB:(i + 1) * NB * NB].reshape((NB, NB), order="F")
            tm, tn = min(NB, N - m * NB), min(NB, N - n * NB)
            t[tm:, :] = np.nan
            t[:, tn:] = np.nan
            if m == n:
                t[np.triu_indices(tm, 1)] = np.nan
    B = rng.uniform(-1.0, 1.0, (N, 3)).astype(dtype)
    dT, dB = dev.upload(T), dev.upload(np.asfortranarray(B).reshape(-1, order="F"))
    fn = dev.M.mi_dtrsm_LL if dtype == np.float64 else dev.M.mi_strsm_LL
    dev.check(fn(dev.h, trans, 132 if unit else 131, 1.0, N, NB, dT, 3, dB, N), "trsm")
    x = dev.download(dB, (N * 3,), dtype).reshape((N, 3), order="F").astype(np.float64)
    dev.free(dT)
    dev.free(dB)
    if unit:
        L[np.diag_indices(N)] = 1.0
    ref = np.linalg.solve(L.T if trans == 112 else L, B.astype(np.float64))
    eps = 2.0 ** -53 if dtype == np.float64 else EPS32
    assert np.abs(x - ref).max() <= 16 * (N + 16) * eps * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("solve", [True, False])
def test_batched_block_edges(dev, dtype, solve):
    """Orders around the 16-column blocks, the size classes (64, 128) and the
    128-column panels, every upper triangle NaN; one matrix without a positive
    pivot in the middle (its right-hand side stays).  G^T G / n + I has a
    condition below 6: n eps times a small factor."""
    ns = [1, 15, 16, 17, 47, 48, 49, 63, 64, 65, 111, 112, 113, 127, 128, 129, 143, 144, 145, 240, 256, 257, 272, 383,
          384, 385, 400, 530, 641, 897, 1009]
    bad = ns.index(145)
    rng = np.random.default_rng(3)
    As, bs = [], []
    for n in ns:
        G = rng.standard_normal((n, n))
        As.append((G.T @ G / n + np.eye(n)).astype(dtype))
        bs.append(rng.uniform(-0.5, 0.5, n).astype(dtype))
    As[bad][130, 130] = -1.0
    flat = []
    for A in As:
        M = A.copy()
        M[np.triu_indices(M.shape[0], 1)] = np.nan
        flat.append(M.ravel(order="F"))
    a, b = np.concatenate(flat), np.concatenate(bs)
    p = ctypes.c_void_p()
    dev.check(dev.M.mi_batch_create(dev.h, len(ns), (ctypes.c_int * len(ns))(*ns), ctypes.byref(p)), "create")
    da, db = dev.upload(a), dev.upload(b)
    fn = dev.M.mi_dposv_batched if dtype == np.float64 else dev.M.mi_sposv_batched
    try:
        dev.check(fn(p, da, db if solve else None, 0), "posv_batched")
        ra, rb = dev.download(da, a.shape, dtype), dev.download(db, b.shape, dtype)
        info = (ctypes.c_int * len(ns))()
        dev.check(dev.M.mi_batch_info(p, info), "info")
    finally:
        dev.M.mi_batch_destroy(p)
        dev.free(da)
        dev.free(db)
    eps = 2.0 ** -53 if dtype == np.float64 else EPS32
    ao = bo = 0
    for i, n in enumerate(ns):
        L, x = ra[ao:ao + n * n].reshape((n, n), order="F"), rb[bo:bo + n]
        assert np.isnan(L[np.triu_indices(n, 1)]).all(), n
        if i == bad:
            assert info[i] == 131 and np.array_equal(x, bs[i])
        else:
            assert info[i] == 0, n
            ref = np.linalg.cholesky(As[i].astype(np.float64))
            assert np.abs(np.tril(L) - ref).max() <= 16 * (n + 16) * eps * np.abs(ref).max(), n
            want = np.linalg.solve(As[i].astype(np.float64), bs[i].astype(np.float64)) if solve else bs[i]
            assert np.abs(x - want).max() <= 64 * (n + 16) * eps * max(1.0, np.abs(want).max()), n
        ao += n * n
        bo += n


@pytest.mark.parametrize("N,NB,dtype", [(3584, 256, np.float64), (4101, 256, np.float64), (4700, 256, np.float64),
                                        (2500, 93, np.float64), (5900, 256, np.float32), (6200, 320, np.float32)])
def test_two_streams_then_one(dev, po, N, NB, dtype):
    """Steps whose updates are large enough for a bulk beside the panels, none
    to several of them, before the ones that run on one stream."""
    A = po.dplgsy_full(N, float(N), 3872).astype(dtype).astype(np.float64)
    ref = np.linalg.cholesky(A)
    for _ in range(2):
        L, info = factor(dev, A, NB, dtype)
        assert info == 0
        assert np.abs(L - ref).max() <= (1e-12 if dtype == np.float64 else 64 * EPS32) * np.abs(ref).max()
    bad = A.copy()
    bad[N - 3, N - 3] = -1.0
    _, info = factor(dev, bad, NB, dtype)
    assert info == N - 2
