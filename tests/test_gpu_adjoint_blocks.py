"""The products of the reverse factorization at the edges of their blocks and
splits: a last tile with a short stage of k, tiles that are no multiple of the
64- or 128-wide blocks, 128-wide blocks over a split k, tiles without whole
stages (FP32: 48; FP64: 200) and an array that is not 16-byte aligned, which
take the general kernel.  Everything outside the lower triangles is NaN.

A = B B^T / N + I has its eigenvalues in [1, 5.2], so the reverse, in which
L^-1 stands on both sides, loses at most a small multiple of N u kappa(A) of
the largest entry: 64 N u."""
import ctypes
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import adjoint as oad  # noqa: E402

from test_gpu_adjoint import pack_lower, unpack_lower  # noqa: E402

pytestmark = pytest.mark.gpu


def at(p):
    return p.value if isinstance(p, ctypes.c_void_p) else int(p)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("N,NB,shift", [(33, 32, 0), (130, 48, 0), (261, 96, 0), (500, 200, 0), (777, 64, 0),
                                        (1500, 160, 0), (3111, 512, 0), (600, 128, 1)])
def test_adjoint_blocks(dev, N, NB, shift, dtype):
    rng = np.random.default_rng(N + NB)
    B = rng.standard_normal((N, N))
    L = np.linalg.cholesky(B @ B.T / N + np.eye(N))
    Lbar = np.tril(rng.standard_normal((N, N)))
    L, Lbar = L.astype(dtype).astype(np.float64), Lbar.astype(dtype).astype(np.float64)
    want = oad.adjoint_closed(L, Lbar)
    pad = np.full(shift, np.nan, dtype)
    size = np.dtype(dtype).itemsize
    dl = dev.upload(np.concatenate([pad, pack_lower(L, NB, dtype=dtype)]))
    G = np.concatenate([pad, pack_lower(Lbar, NB, dtype=dtype)])
    dg = dev.upload(G)
    fn = dev.M.mi_dpotrf_adjoint_tiles if dtype == np.float64 else dev.M.mi_spotrf_adjoint_tiles
    dev.check(fn(dev.h, N, NB, ctypes.c_void_p(at(dl) + shift * size), ctypes.c_void_p(at(dg) + shift * size)), "adjoint")
    got = dev.download(dg, G.shape, dtype)[shift:]
    dev.free(dl)
    dev.free(dg)
    got, outside = unpack_lower(got, N, NB)
    assert np.isnan(outside).all()
    tol = 64 * N * np.finfo(dtype).eps
    assert np.abs(np.tril(got) - np.tril(want)).max() <= tol * np.abs(want).max()
