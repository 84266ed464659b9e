"""Calls of a batch plan in any order, and what a plan's first call costs."""
import ctypes
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Plan:
    def __init__(self, dev, ns):
        self.dev, self.ns, self.p = dev, ns, ctypes.c_void_p()
        dev.check(dev.M.mi_batch_create(dev.h, len(ns), (ctypes.c_int * len(ns))(*ns), ctypes.byref(self.p)), "create")

    def close(self):
        self.dev.M.mi_batch_destroy(self.p)


def systems(ns, dtype):
    rng = np.random.default_rng(len(ns))
    a = []
    for n in ns:
        g = 0.2 * rng.standard_normal((n, n)) / n
        a.append((g + g.T + 2.0 * np.eye(n)).ravel())
    return np.concatenate(a).astype(dtype), rng.uniform(-0.5, 0.5, sum(ns)).astype(dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("ns", [[5], [70] * 3, [200, 130], [300, 100, 20, 1], [90, 60, 64, 65], [250, 64, 3]],
                         ids=lambda v: "-".join(map(str, v)))
def test_every_call_finds_its_queue_empty(dev, ns, dtype):
    """Direct calls, graphs, launch loops, other arrays and other numbers of
    workgroups one after the other: every result is that of the first call,
    bit for bit."""
    a, b = systems(ns * 20, dtype)
    f = "d" if dtype == np.float64 else "s"
    run, loop = getattr(dev.M, f"mi_{f}posv_batched"), getattr(dev.M, f"mi_{f}posv_batched_loop")
    plan = Plan(dev, ns * 20)
    arrays = [(dev.upload(a), dev.upload(b)) for _ in range(2)]
    want = None
    try:
        for step, (which, kind, wg) in enumerate([(0, "direct", 2), (0, "graph", 2), (0, "graph", 2), (1, "graph", 2),
                                                  (1, "loop", 2), (0, "direct", 1), (0, "graph", 1), (1, "loop", 1),
                                                  (0, "graph", 1), (0, "factor", 2), (1, "graph", 2)]):
            da, db = arrays[which]
            dev.check(dev.M.mi_memcpy_h2d(dev.h, da, a.ctypes.data, a.nbytes), "h2d")
            dev.check(dev.M.mi_memcpy_h2d(dev.h, db, b.ctypes.data, b.nbytes), "h2d")
            dev.check(dev.M.mi_batch_set_shape(plan.p, 128, wg), "shape")
            if kind == "loop":
                dev.check(loop(plan.p, da, db), "loop")
            else:
                dev.check(run(plan.p, da, None if kind == "factor" else db, int(kind == "graph")), kind)
            ra, rb = dev.download(da, a.shape, dtype), dev.download(db, b.shape, dtype)
            want = want or (ra, rb)
            assert np.array_equal(ra, want[0]), (step, kind)
            assert np.array_equal(rb, b if kind == "factor" else want[1]), (step, kind)
    finally:
        plan.close()
        for da, db in arrays:
            dev.free(da)
            dev.free(db)


def first_call_extra(dev, ns):
    """What the first call of a plan costs more than the next ones, us (medians of 15 plans)."""
    a, b = systems(ns, np.float32)
    da, db = dev.upload(a), dev.upload(b)
    first, later = [], []
    for _ in range(15):
        plan = Plan(dev, ns)
        for times in (first, later, later):
            dev.check(dev.M.mi_memcpy_h2d(dev.h, da, a.ctypes.data, a.nbytes), "h2d")
            dev.check(dev.M.mi_memcpy_h2d(dev.h, db, b.ctypes.data, b.nbytes), "h2d")
            t = time.perf_counter()
            dev.check(dev.M.mi_sposv_batched(plan.p, da, db, 1), "batched")
            times.append((time.perf_counter() - t) * 1e6)
        plan.close()
    dev.free(da)
    dev.free(db)
    return float(np.median(first) - np.median(later))


def test_first_call_captures_one_launch(dev):
    """With use_graph a plan's first call captures one launch, whether its
    matrices are of one size class or of several: what it costs beyond a
    replay is the same, up to a factor of 3 for the clock's noise (a graph with
    a branch for the smaller classes: 5 to 10 times as much)."""
    rng = np.random.default_rng(5)
    first_call_extra(dev, [10] * 64)                             # the process's first capture
    one = first_call_extra(dev, rng.integers(1, 65, 64).tolist())
    several = first_call_extra(dev, rng.integers(1, 201, 64).tolist())
    print(f"one class {one:.1f} us, several {several:.1f} us")
    assert several <= 3.0 * one
