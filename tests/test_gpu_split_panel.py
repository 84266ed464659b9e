"""The BF16-split FP32 factor with its panel columns split once per step, at
sizes where that path runs: steps whose whole update exceeds 2^31 FP64-sized
multiply-adds (NB^3 / 4 of them a tile in FP32), with tiles that are no
multiple of the 256- or 128-row blocks and ragged last tiles.  The profiler's
kernel names say that it ran."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(8700, 128), (6300, 320), (5600, 384), (5000, 448)]


def factor(dev, T, N, NB, which):
    """The factor's tiles, and the launches of the splitting kernel."""
    M = dev.M
    d = dev.upload(T)
    info, n = ctypes.c_int(-1), ctypes.c_int(0)
    ms, fl, by = ctypes.c_double(), ctypes.c_double(), ctypes.c_double()
    dev.check(M.mi_set_spotrf_update(1), "bf16x3")
    dev.check(M.mi_set_bf16_panel_split(which), "panel split")
    try:
        M.mi_prof_enable(dev.h, 1)
        M.mi_prof_reset(dev.h)
        dev.check(M.mi_spotrf_tiles(dev.h, N, NB, d, ctypes.byref(info)), "spotrf")
        names = {M.mi_prof_name(dev.h, i).decode() for i in range(M.mi_prof_count(dev.h))}
        if "spotrf_split_panel" in names:
            M.mi_prof_get(dev.h, b"spotrf_split_panel", *map(ctypes.byref, (n, ms, fl, by)))
        return dev.download(d, T.shape, np.float32), info.value, n.value
    finally:
        M.mi_prof_enable(dev.h, 0)
        M.mi_set_spotrf_update(0)
        M.mi_set_bf16_panel_split(1)
        dev.free(d)


@pytest.mark.parametrize("N,NB", SIZES)
def test_split_once_gives_the_same_factor(dev, po, N, NB):
    print(f"split panel N={N} NB={NB}", flush=True)
    T = po.dplgsy_symtiles(N, NB, float(N), 3872).astype(np.float32)
    MT = (N + NB - 1) // NB
    steps = sum((MT - k - 1) * (MT - k) * 0.25 * NB ** 3 > 2.0 ** 31 for k in range(MT - 2))
    assert steps > 0
    a, ia, na = factor(dev, T, N, NB, 0)
    b, ib, nb = factor(dev, T, N, NB, 1)
    assert ia == ib == 0 and na == 0 and nb == steps
    assert np.array_equal(a, b)


@pytest.mark.parametrize("N,NB", SIZES[1:])
def test_split_factor_against_fp64(dev, po, N, NB):
    """The split keeps 16 bits of each operand and each of the MT steps adds
    one update: MT 2^-16 of the largest entry."""
    print(f"split factor N={N} NB={NB}", flush=True)
    T = po.dplgsy_symtiles(N, NB, float(N), 3872).astype(np.float32)
    got, info, n = factor(dev, T, N, NB, 1)
    assert info == 0 and n > 0
    low = lambda t: np.tril(po.symtiles_to_full(t.astype(np.float64), N, NB))
    A = low(T)
    ref = np.linalg.cholesky(A + np.tril(A, -1).T)
    assert np.abs(low(got) - ref).max() <= (N + NB - 1) // NB * 2.0 ** -16 * np.abs(ref).max()
