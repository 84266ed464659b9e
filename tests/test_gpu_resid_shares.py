"""The symmetric residual with one and with several workgroups a tile, its
norm of A, and the number of workgroups it takes.

A sum of N products and one term, added up in any order, is within
(N + 1) u (|A| |X| + |B|) of the exact one, element by element; numpy's FP64
reference adds as much."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def tiles(po, A, NB):
    """Packed lower tiles, NaN in every element that must not be read."""
    N = A.shape[0]
    T, MT = po.full_to_symtiles(A, NB), (N + NB - 1) // NB
    for n in range(MT):
        for m in range(n, MT):
            i = n * MT - n * (n - 1) // 2 + (m - n)
            t = T[i * NB * NB:(i + 1) * NB * NB].reshape((NB, NB), order="F")
            tm, tn = min(NB, N - m * NB), min(NB, N - n * NB)
            t[tm:, :] = np.nan
            t[:, tn:] = np.nan
            if m == n:
                t[np.triu_indices(tm, 1)] = np.nan
    return T


# 253 to 300 tiles: one workgroup a tile, but for NB = 90 with few right-hand
# sides; the others share theirs
@pytest.mark.parametrize("kernel", [1, 0], ids=["lds_chunks", "registers"])
@pytest.mark.parametrize("nrhs", [1, 3, 8, 16, 20])
@pytest.mark.parametrize("N,NB", [(1500, 64), (2900, 128), (1980, 90), (900, 320), (1100, 512), (1900, 256)])
def test_residual_and_norm(dev, po, N, NB, nrhs, kernel):
    print(f"resid N={N} NB={NB} nrhs={nrhs} kernel={kernel}", flush=True)
    rng = np.random.default_rng(N)
    A = rng.standard_normal((N, N))
    A = A + A.T
    X, B = rng.standard_normal((N, nrhs)), rng.standard_normal((N, nrhs))
    cm = lambda M: dev.upload(np.asfortranarray(M).reshape(-1, order="F"))
    dT, dX, dB, dR = dev.upload(tiles(po, A, NB)), cm(X), cm(B), dev.alloc(N * nrhs * 8)
    norms = [ctypes.c_double(-1.0) for _ in range(4)]
    try:
        dev.check(dev.M.mi_set_symm_kernel(kernel), "symm kernel")
        dev.check(dev.M.mi_dsymm_resid(dev.h, N, NB, dT, nrhs, dX, N, dB, N, dR, N), "resid")
        dev.check(dev.M.mi_dcheck_axmb(dev.h, N, NB, dT, nrhs, dB, N, dX, N, *map(ctypes.byref, norms)), "check")
    finally:
        dev.M.mi_set_symm_kernel(1)
    R = dev.download(dR, (N * nrhs,)).reshape((N, nrhs), order="F")
    for p in (dT, dX, dB, dR):
        dev.free(p)
    tol = 2 * (N + 1) * U * (np.abs(A) @ np.abs(X) + np.abs(B))
    assert (np.abs(R - (B - A @ X)) <= tol).all()
    norm = np.abs(A).sum(axis=1).max()
    assert abs(norms[0].value - norm) <= 2 * N * U * norm


@pytest.mark.parametrize("N,NB,nrhs,most,least", [(4096, 256, 1, 3, 3), (4096, 256, 16, 1, 1), (2000, 100, 16, 1, 1),
                                                  (1000, 128, 16, 1, 1), (3200, 320, 16, 6, 3), (4096, 512, 16, 6, 3),
                                                  (10000, 512, 16, 1, 1)])
def test_workgroups_a_tile(dev, N, NB, nrhs, most, least):
    """Where sharing a tile makes the sum of the partials longer than the
    products become shorter, it is not shared (measured best: N = 4096, NB =
    256, 16 right-hand sides 63 us unshared, 80 with two).  The profiler's
    bytes of the sum, 8 (S + 1) NB 16 a tile, tell the number S."""
    MT = (N + NB - 1) // NB
    nt = MT * (MT + 1) // 2
    d = dev.alloc(nt * NB * NB * 8)
    v = dev.alloc(3 * N * nrhs * 8)
    M = dev.M
    dev.check(M.mi_memset(dev.h, d, 0, nt * NB * NB * 8), "memset")
    dev.check(M.mi_memset(dev.h, v, 0, 3 * N * nrhs * 8), "memset")
    n, ms, fl, by = ctypes.c_int(), ctypes.c_double(), ctypes.c_double(), ctypes.c_double()
    try:
        M.mi_prof_enable(dev.h, 1)
        M.mi_prof_reset(dev.h)
        dev.check(M.mi_dsymm_resid(dev.h, N, NB, d, nrhs, v, N, v + N * nrhs * 8, N, v + 2 * N * nrhs * 8, N), "resid")
        M.mi_prof_get(dev.h, b"dsymm_sum", *map(ctypes.byref, (n, ms, fl, by)))
    finally:
        M.mi_prof_enable(dev.h, 0)
        dev.free(d)
        dev.free(v)
    S = by.value / (8 * 16 * nt * NB) - 1
    print(f"N={N} NB={NB} nrhs={nrhs}: S={S}")
    assert n.value == 1 and least <= S <= most
