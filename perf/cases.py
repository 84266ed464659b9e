"""Timed cases of the tile Cholesky factor-and-solve library.

Each case is one call (or one forward and backward pass) that a program using
this library makes, over the sizes, tile sizes, precisions and options it is
used with: the tile factorization and solve on tiles in device memory, the
LAPACK-layout solve, the mixed-precision solve on device tiles and through
the host descriptors of the dplasma interface, the batched solve of many
small systems, and the Gaussian-process likelihood with its gradient.

Input values: matrices that are factored alone are those of dplasma_dplgsy
(entries uniform in [-1/2, 1/2), bump N on the diagonal); systems that are
solved are squared-exponential kernel matrices with noise, of a condition
below about 1e2 where FP32 takes part and a few 1e3 otherwise; the batch is
G^T G / n + I, as the batched benchmark's.
"""
import ctypes
import math

import numpy as np
import torch

import dplasma_amd as dp
import dplasma_amd.autograd as ag

DTYPES = {"f64": torch.float64, "f32": torch.float32}
BYTES = {"f64": 8, "f32": 4}


# ------------------------------------------------------------------ cases
def listed():
    return [
        # The reference's headline problem: one large FP64 factorization, tiles resident.
        {"name": "potrf_f64_32768", "kind": "potrf", "dtype": "f64", "N": 32768, "NB": 512},
        # The reference's CPU-sized benchmark: 16 steps, ordinary size.
        {"name": "potrf_f64_4096", "kind": "potrf", "dtype": "f64", "N": 4096, "NB": 256},
        # The smallest factorization of the reference's test list, odd tile size, ragged last tile.
        {"name": "potrf_f64_378", "kind": "potrf", "dtype": "f64", "N": 378, "NB": 93},
        # A single-precision factorization (the preconditioner of a user's own iteration), ragged.
        {"name": "potrf_f32_10000", "kind": "potrf", "dtype": "f32", "N": 10000, "NB": 512},
        # Solve with a factor that is kept, one right-hand side: a time step of an implicit scheme.
        {"name": "potrs_f64_32768_1", "kind": "potrs", "N": 32768, "NB": 512, "nrhs": 1},
        # Mixed-precision solve to FP64 backward error, the large configuration with the BF16-split factor.
        {"name": "mixed_bf16_32768", "kind": "mixed", "prec": "bf16x3", "N": 32768, "NB": 512, "nrhs": 16},
        # The same through the host descriptors (dplasma_dposv_mixed), FP32 factor, a size of the test list.
        {"name": "mixed_host_3200", "kind": "host", "prec": "f32", "N": 3200, "NB": 320, "nrhs": 1},
        # Factor and solve of a caller's column-major array, upper triangle, odd leading dimension, ragged.
        {"name": "posv_lapack_6000", "kind": "lapack", "uplo": "U", "N": 6000, "NB": 512, "nrhs": 4, "lda": 6001},
        # Many uneven systems at once, the batched benchmark's sizes.
        {"name": "batch_f64_4096", "kind": "batch", "dtype": "f64", "count": 4096, "lo": 32, "hi": 1024},
        # A batch of small systems in single precision (per-cell or per-voxel solves).
        {"name": "batch_f32_1000", "kind": "batch", "dtype": "f32", "count": 1000, "lo": 8, "hi": 200},
        # Likelihood and gradient of one Gaussian process on 8192 points, forward and backward.
        {"name": "gp_f64_8192", "kind": "gp", "dtype": "f64", "N": 8192, "NB": 512},
        # One of the many small processes of a batch of fits, single precision.
        {"name": "gp_f32_1024", "kind": "gp", "dtype": "f32", "N": 1024, "NB": 256},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _nb(rng, N):
    """Tile sizes in use: the test list's odd ones for small matrices, multiples of 32 beyond."""
    if N <= 4000:
        return rng.choice([93, 128, 160, 200, 256, 320, 367, 512])
    return rng.choice([256, 320, 384, 512, 512])


def draw(rng):
    kind = rng.choice(["potrf", "potrf", "potrf", "potrs", "mixed", "host", "lapack", "batch", "batch", "gp", "gp"])
    if kind == "potrf":
        N = _log(rng, 200, 28000)
        return {"kind": kind, "dtype": rng.choice(["f64", "f64", "f32"]), "N": N, "NB": _nb(rng, N)}
    if kind == "potrs":
        N = _log(rng, 500, 32768)
        return {"kind": kind, "N": N, "NB": _nb(rng, N), "nrhs": _log(rng, 1, 40)}
    if kind == "mixed":
        N = _log(rng, 2000, 28000)
        return {"kind": kind, "prec": rng.choice(["f32", "bf16x3"]), "N": N, "NB": rng.choice([256, 320, 384, 512]),
                "nrhs": _log(rng, 1, 32)}
    if kind == "host":
        N = _log(rng, 300, 8000)
        return {"kind": kind, "prec": rng.choice(["f32", "bf16x3"]), "N": N, "NB": _nb(rng, N), "nrhs": _log(rng, 1, 8)}
    if kind == "lapack":
        N = _log(rng, 300, 16000)
        return {"kind": kind, "uplo": rng.choice(["L", "U"]), "N": N, "NB": rng.choice([256, 512]),
                "nrhs": _log(rng, 1, 16), "lda": N + rng.randrange(0, 9)}
    if kind == "batch":
        lo = _log(rng, 1, 64)
        hi = min(1024, lo + _log(rng, 16, 960))
        count = _log(rng, 64, 4096)
        return {"kind": kind, "dtype": rng.choice(["f64", "f32"]), "count": count, "lo": lo, "hi": hi}
    N = _log(rng, 300, 12000)
    return {"kind": "gp", "dtype": rng.choice(["f64", "f32"]), "N": N, "NB": rng.choice([256, 512])}


# ------------------------------------------------------------------ handles
class _Handles:
    device = None
    context = None


def _device():
    """The kernel context of this process (one per GPU, kept)."""
    if _Handles.device is None:
        _Handles.device = dp.Device(torch.cuda.current_device())
    return _Handles.device


def _context():
    """The dplasma context of this process."""
    if _Handles.context is None:
        _Handles.context = dp.Context(torch.cuda.current_device())
    return _Handles.context


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _ready():
    """The library works on streams of its own: what torch queued has to be done."""
    torch.cuda.current_stream().synchronize()


class _Plan:
    """A batch plan (mi_batch_create), given back with the state."""

    def __init__(self, ns):
        d = _device()
        self.count = len(ns)
        self.p = ctypes.c_void_p()
        d.check(d.M.mi_batch_create(d.h, self.count, (ctypes.c_int * self.count)(*ns), ctypes.byref(self.p)),
                "mi_batch_create")

    def __del__(self):
        _device().M.mi_batch_destroy(self.p)


# ------------------------------------------------------------------ inputs
def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 64 + salt)
    return g


def _tile_order(N, NB):
    MT = (N + NB - 1) // NB
    return MT, [(m, n) for n in range(MT) for m in range(n, MT)]


def _spd_tiles(N, NB, seed, dtype):
    """dplgsy-like packed lower tiles ([tile][column][row]): full diagonal tiles, zero padding rows."""
    MT, order = _tile_order(N, NB)
    T = torch.rand((len(order), NB, NB), generator=_gen(seed, 0), device="cuda", dtype=dtype)
    T -= 0.5
    last = N - (MT - 1) * NB
    at = 0
    for n in range(MT):
        D = T[at]
        D.copy_(D.tril() + D.tril(-1).T)
        D.diagonal().add_(float(N))
        at += MT - n
        T[at - 1, :, last:] = 0.0
    T[-1, last:, :] = 0.0
    return T


def _factor_tiles(N, NB, seed):
    """The factor of such a matrix: diagonal sqrt(N), entries of size 1 / sqrt(N) below it."""
    MT, order = _tile_order(N, NB)
    T = torch.rand((len(order), NB, NB), generator=_gen(seed, 0), device="cuda", dtype=torch.float64)
    T -= 0.5
    T /= math.sqrt(N)
    last = N - (MT - 1) * NB
    at = 0
    for n in range(MT):
        T[at].diagonal().fill_(math.sqrt(N))
        at += MT - n
        T[at - 1, :, last:] = 0.0
    T[-1, last:, :] = 0.0
    return T


def _points(N, seed):
    return torch.rand((N, 3), generator=_gen(seed, 1), device="cuda", dtype=torch.float64)


def _lengthscale(N):
    """About 20 points within reach of each point of the unit cube (the largest eigenvalue)."""
    return (20.0 / N) ** (1.0 / 3.0) / math.sqrt(2.0 * math.pi)


def _se_block(X, r0, r1, c0, c1, noise):
    l = _lengthscale(X.shape[0])
    d2 = torch.zeros((r1 - r0, c1 - c0), device="cuda", dtype=torch.float64)
    for k in range(3):
        d2 += (X[r0:r1, k, None] - X[None, c0:c1, k]) ** 2
    K = torch.exp(d2 * (-0.5 / (l * l)))
    if r0 == c0:
        K.diagonal().add_(noise)
    return K


def _se_tiles(N, NB, seed, noise):
    """Squared-exponential kernel matrix in packed lower tiles."""
    X = _points(N, seed)
    MT, order = _tile_order(N, NB)
    T = torch.zeros((len(order), NB, NB), device="cuda", dtype=torch.float64)
    at = 0
    for n in range(MT):
        c0, c1 = n * NB, min(N, (n + 1) * NB)
        col = torch.zeros(((MT - n) * NB, NB), device="cuda", dtype=torch.float64)
        col[:N - c0, :c1 - c0] = _se_block(X, c0, N, c0, c1, noise)
        T[at:at + MT - n] = col.view(MT - n, NB, NB).transpose(1, 2)
        at += MT - n
    return T


def _se_dense(N, seed, noise):
    X = _points(N, seed)
    K = torch.empty((N, N), device="cuda", dtype=torch.float64)
    for c0 in range(0, N, 1024):
        c1 = min(N, c0 + 1024)
        K[c0:, c0:c1] = _se_block(X, c0, N, c0, c1, noise)
        K[c0:c1, c1:] = K[c1:, c0:c1].T
    return K


def _rhs(N, nrhs, seed):
    """Column-major right-hand sides as an (nrhs, N) array."""
    return torch.rand((nrhs, N), generator=_gen(seed, 2), device="cuda", dtype=torch.float64) - 0.5


def _sizes(case):
    """The orders of a batch: a program's plan, the same for every set of inputs."""
    rng = np.random.default_rng([case["count"], case["lo"], case["hi"]])
    return rng.integers(case["lo"], case["hi"] + 1, case["count"]).tolist()


def _batch_inputs(case, seed):
    ns = _sizes(case)
    dt = DTYPES[case["dtype"]]
    total = sum(n * n for n in ns)
    A = torch.empty(total, device="cuda", dtype=dt)
    G = torch.randn(total, generator=_gen(seed, 0), device="cuda", dtype=dt)
    at = 0
    for n in ns:
        g, a = G[at:at + n * n].view(n, n), A[at:at + n * n].view(n, n)
        torch.mm(g.T, g, out=a)
        a /= n
        a.diagonal().add_(1.0)
        at += n * n
    b = torch.rand(sum(ns), generator=_gen(seed, 2), device="cuda", dtype=dt) - 0.5
    return ns, A, b


NOISE = {"f64": 1e-2, "f32": 1.0, "mixed": 0.5}


def prepare(case, seed):
    kind = case["kind"]
    N, NB = case.get("N"), case.get("NB")
    s = {"case": dict(case)}
    if kind == "potrf":
        s["A0"] = _spd_tiles(N, NB, seed, DTYPES[case["dtype"]])
        s["A"] = torch.empty_like(s["A0"])
    elif kind == "potrs":
        s["L"] = _factor_tiles(N, NB, seed)
        s["B"] = _rhs(N, case["nrhs"], seed)
        s["X"] = torch.empty_like(s["B"])
    elif kind == "mixed":
        s["A"] = _se_tiles(N, NB, seed, NOISE["mixed"])
        s["B"] = _rhs(N, case["nrhs"], seed)
        s["X"] = torch.empty_like(s["B"])
    elif kind == "host":
        ctx = _context()
        s["A"] = dp.SymMatrix(ctx, N, NB, dp.LOWER)
        s["A"].array[:] = _se_tiles(N, NB, seed, NOISE["mixed"]).reshape(-1).cpu().numpy()
        s["B"] = dp.GeMatrix(ctx, N, case["nrhs"], NB, NB)
        s["B"].from_numpy(_rhs(N, case["nrhs"], seed).T.cpu().numpy())
        s["X"] = dp.GeMatrix(ctx, N, case["nrhs"], NB, NB)
    elif kind == "lapack":
        s["A0"] = torch.zeros((N, case["lda"]), device="cuda", dtype=torch.float64)
        s["A0"][:, :N] = _se_dense(N, seed, NOISE["f64"])
        s["B0"] = _rhs(N, case["nrhs"], seed)
        s["A"], s["B"] = torch.empty_like(s["A0"]), torch.empty_like(s["B0"])
    elif kind == "batch":
        ns, s["A0"], s["B0"] = _batch_inputs(case, seed)
        s["A"], s["B"] = torch.empty_like(s["A0"]), torch.empty_like(s["B0"])
        s["plan"] = _Plan(ns)
    else:
        dt = DTYPES[case["dtype"]]
        s["K"] = _se_dense(N, seed, NOISE[case["dtype"]]).to(dt).requires_grad_(True)
        s["y"] = torch.randn(N, generator=_gen(seed, 2), device="cuda", dtype=torch.float64).to(dt)
    return s


# ------------------------------------------------------------------ one pass
PREC = {"f32": dp.MIXED_FP32, "bf16x3": dp.MIXED_BF16X3}


def run(s):
    case = s["case"]
    kind, N, NB = case["kind"], case.get("N"), case.get("NB")
    d = _device()
    info = ctypes.c_int(-1)
    if kind == "potrf":
        # the factorization overwrites its input: a program that keeps the matrix copies it first
        s["A"].copy_(s["A0"])
        _ready()
        fn = d.M.mi_dpotrf_tiles if case["dtype"] == "f64" else d.M.mi_spotrf_tiles
        d.check(fn(d.h, N, NB, _p(s["A"]), ctypes.byref(info)), "potrf")
        return {"L": s["A"], "info": info.value}
    if kind == "potrs":
        s["X"].copy_(s["B"])
        _ready()
        d.check(d.M.mi_dpotrs_tiles(d.h, N, NB, _p(s["L"]), case["nrhs"], _p(s["X"]), N), "potrs")
        return {"X": s["X"]}
    if kind == "mixed":
        it = ctypes.c_int(0)
        _ready()
        d.check(d.M.mi_dsposv_tiles(d.h, N, NB, _p(s["A"]), case["nrhs"], _p(s["B"]), N, _p(s["X"]), N,
                                    PREC[case["prec"]], ctypes.byref(it), ctypes.byref(info)), "dsposv")
        return {"X": s["X"], "info": info.value}
    if kind == "host":
        rc, _ = _context().dposv_mixed(dp.LOWER, s["A"], s["B"], s["X"], PREC[case["prec"]])
        return {"X": s["X"].to_numpy(), "info": rc}
    if kind == "lapack":
        s["A"].copy_(s["A0"])
        s["B"].copy_(s["B0"])
        _ready()
        uplo = dp.UPPER if case["uplo"] == "U" else dp.LOWER
        d.check(d.M.mi_dposv_lapack(d.h, uplo, N, case["nrhs"], _p(s["A"]), case["lda"], _p(s["B"]), N, NB,
                                    ctypes.byref(info)), "posv_lapack")
        return {"A": s["A"], "X": s["B"], "info": info.value}
    if kind == "batch":
        s["A"].copy_(s["A0"])
        s["B"].copy_(s["B0"])
        _ready()
        fn = d.M.mi_dposv_batched if case["dtype"] == "f64" else d.M.mi_sposv_batched
        d.check(fn(s["plan"].p, _p(s["A"]), _p(s["B"]), 1), "posv_batched")
        return {"A": s["A"], "X": s["B"]}
    s["K"].grad = None
    nll = ag.gp_nll(s["K"], s["y"], NB)
    nll.backward()
    return {"nll": nll.detach(), "dK": s["K"].grad}


# ------------------------------------------------------------------ least work
def _tri_solve(N, nrhs):
    return 2.0 * N * N * nrhs


def work(case):
    kind = case["kind"]
    if kind == "batch":
        # the lower triangles read and written, the right-hand sides too
        n = np.array(_sizes(case), dtype=np.float64)
        n2, n3 = (n ** 2).sum(), (n ** 3).sum()
        return {"bytes": BYTES[case["dtype"]] * (n2 + 3.0 * n.sum()), "flops": n3 / 3.0 + 2.0 * n2}
    N, r = float(case["N"]), float(case.get("nrhs", 0))
    tri = N * (N + 1.0) / 2.0
    chol = N ** 3 / 3.0
    if kind == "potrf":
        return {"bytes": 2.0 * tri * BYTES[case["dtype"]], "flops": chol}
    if kind == "potrs":
        return {"bytes": 8.0 * (tri + 2.0 * N * r), "flops": _tri_solve(N, r)}
    if kind in ("mixed", "host"):
        # A is read once; one refinement step at least: two solves and two residuals
        return {"bytes": 8.0 * (tri + 2.0 * N * r), "flops": chol + 2.0 * (_tri_solve(N, r) + 2.0 * N * N * r)}
    if kind == "lapack":
        return {"bytes": 8.0 * (2.0 * tri + 2.0 * N * r), "flops": chol + _tri_solve(N, r)}
    # factor (N^3 / 3) and its reverse (2 N^3 / 3), one solve; K read, its gradient written
    return {"bytes": BYTES[case["dtype"]] * 2.0 * N * N, "flops": N ** 3 + N * N}


# ------------------------------------------------------------------ in 64 bits, by torch
def _dense_lower(T, N, NB):
    """Packed lower tiles -> dense, the lower triangle filled."""
    MT, _ = _tile_order(N, NB)
    D = torch.zeros((MT * NB, MT * NB), device="cuda", dtype=torch.float64)
    at = 0
    for n in range(MT):
        D[n * NB:, n * NB:(n + 1) * NB] = T[at:at + MT - n].transpose(1, 2).reshape((MT - n) * NB, NB).double()
        at += MT - n
    return D[:N, :N]


def _into_tiles(L, T, N, NB):
    """Dense lower triangle -> a copy of the tiles T; what the factorization leaves alone stays."""
    MT, _ = _tile_order(N, NB)
    R = T.double()
    at = 0
    for n in range(MT):
        c0, c1 = n * NB, min(N, (n + 1) * NB)
        for m in range(n, MT):
            r0, r1 = m * NB, min(N, (m + 1) * NB)
            view = R[at, :c1 - c0, :r1 - r0]           # [column][row]
            blk = L[r0:r1, c0:c1].T
            if m == n:
                view.copy_(torch.triu(blk) + torch.tril(view, -1))
            else:
                view.copy_(blk)
            at += 1
    return R


def _exact_batch(case, seed):
    ns, A, b = _batch_inputs(case, seed)
    A, b = A.double(), b.double()
    ao = np.concatenate([[0], np.cumsum(np.square(ns))])
    bo = np.concatenate([[0], np.cumsum(ns)])
    order = sorted(range(len(ns)), key=lambda i: ns[i])
    for g in range(0, len(order), 256):          # neighbours in size together, padded with the identity
        idx = order[g:g + 256]
        n = ns[idx[-1]]
        P = torch.eye(n, device="cuda", dtype=torch.float64).repeat(len(idx), 1, 1)
        q = torch.zeros((len(idx), n, 1), device="cuda", dtype=torch.float64)
        for j, i in enumerate(idx):
            k = ns[i]
            P[j, :k, :k] = A[ao[i]:ao[i + 1]].view(k, k)
            q[j, :k, 0] = b[bo[i]:bo[i + 1]]
        L = torch.linalg.cholesky(P)
        x = torch.linalg.solve_triangular(L, q, upper=False)
        x = torch.linalg.solve_triangular(L.transpose(1, 2).contiguous(), x, upper=True)
        for j, i in enumerate(idx):
            k = ns[i]
            a = A[ao[i]:ao[i + 1]].view(k, k)    # [column][row]: its upper part is the lower triangle
            a.copy_(L[j, :k, :k].T + torch.tril(a, -1))
            b[bo[i]:bo[i + 1]] = x[j, :k, 0]
    return {"A": A, "X": b}


def exact(case, seed):
    kind, N, NB = case["kind"], case.get("N"), case.get("NB")
    if kind == "potrf":
        T = _spd_tiles(N, NB, seed, DTYPES[case["dtype"]])
        D = _dense_lower(T, N, NB)
        return {"L": _into_tiles(torch.linalg.cholesky(D), T, N, NB), "info": None}
    if kind == "potrs":
        L = torch.tril(_dense_lower(_factor_tiles(N, NB, seed), N, NB))
        X = torch.linalg.solve_triangular(L, _rhs(N, case["nrhs"], seed).T.contiguous(), upper=False)
        return {"X": torch.linalg.solve_triangular(L.T, X, upper=True).T.contiguous()}
    if kind in ("mixed", "host"):
        L = torch.linalg.cholesky(_se_dense(N, seed, NOISE["mixed"]))
        X = torch.cholesky_solve(_rhs(N, case["nrhs"], seed).T.contiguous(), L)
        return {"X": X if kind == "host" else X.T.contiguous(), "info": None}
    if kind == "lapack":
        K = _se_dense(N, seed, NOISE["f64"])
        L = torch.linalg.cholesky(K)
        X = torch.cholesky_solve(_rhs(N, case["nrhs"], seed).T.contiguous(), L)
        A = torch.zeros((N, case["lda"]), device="cuda", dtype=torch.float64)     # [column][row]
        if case["uplo"] == "L":
            A[:, :N] = L.T + torch.tril(K, -1)
        else:
            A[:, :N] = L + torch.triu(K, 1)
        return {"A": A, "X": X.T.contiguous(), "info": None}
    if kind == "batch":
        return _exact_batch(case, seed)
    dt = DTYPES[case["dtype"]]
    K = _se_dense(N, seed, NOISE[case["dtype"]]).to(dt).double()
    y = torch.randn(N, generator=_gen(seed, 2), device="cuda", dtype=torch.float64).to(dt).double()
    L = torch.linalg.cholesky(K)
    a = torch.cholesky_solve(y[:, None], L)
    nll = 0.5 * (y @ a[:, 0]) + torch.log(torch.diagonal(L)).sum() + 0.5 * N * math.log(2 * math.pi)
    dK = torch.cholesky_inverse(L)
    dK = 0.5 * (0.5 * (dK + dK.T) - a @ a.T)
    return {"nll": nll, "dK": dK}
