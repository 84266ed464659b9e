"""Differentiable Cholesky for PyTorch over the C ABI of libdplasma_mi.so.

forward:  mi_dpotrf_tiles / mi_spotrf_tiles (the tile factorization),
backward: mi_dpotrf_adjoint_tiles / mi_spotrf_adjoint_tiles (its blocked
          reverse), returning the symmetric gradient with respect to A.

A thin wrapper: dense N x N device tensors are packed into the lower tile
layout of the kernels (tile (m, n), m >= n, column by column, each NB x NB
column-major) and back by the library's staging kernels; the kernels run on
the library's own streams, so the wrapper synchronizes the device around each
call.  With recompute=True only A is kept for the backward pass and L is
factored again there (for when memory is short); otherwise the factor's tiles
are kept.  The backward passes run outside autograd and refuse to be
differentiated themselves.
"""
import ctypes
import math

import torch
from torch.autograd.function import once_differentiable

from . import Device


class _Layout:
    """Index tensors of the packed lower tile order for one (N, NB, device)."""

    _cache = {}

    @classmethod
    def get(cls, N, NB, device):
        key = (N, NB, str(device))
        if key not in cls._cache:
            MT = (N + NB - 1) // NB
            ns = [n for n in range(MT) for m in range(n, MT)]
            ms = [m for n in range(MT) for m in range(n, MT)]
            cls._cache[key] = (MT, torch.tensor(ns, device=device), torch.tensor(ms, device=device))
        return cls._cache[key]


def to_tiles(A, NB):
    """Dense (N x N) -> packed lower tiles (ntiles, NB, NB), tile [column][row]."""
    N = A.shape[0]
    MT, ns, ms = _Layout.get(N, NB, A.device)
    P = MT * NB
    if P != N:
        Ap = A.new_zeros(P, P)
        Ap[:N, :N] = A
    else:
        Ap = A.contiguous()
    T4 = Ap.view(MT, NB, MT, NB).permute(2, 0, 3, 1)     # [n][m][column][row]
    return T4[ns, ms].contiguous()


def from_tiles(T, N, NB):
    """Packed lower tiles -> dense lower triangle (N x N)."""
    MT, ns, ms = _Layout.get(N, NB, T.device)
    T4 = T.new_zeros(MT, MT, NB, NB)
    T4[ns, ms] = T
    return T4.permute(1, 3, 0, 2).reshape(MT * NB, MT * NB)[:N, :N].tril()


class _Lib:
    dev = None

    @classmethod
    def get(cls):
        if cls.dev is None:
            cls.dev = Device(torch.cuda.current_device())
        return cls.dev


def _potrf(T, N, NB):
    d = _Lib.get()
    info = ctypes.c_int(-1)
    fn = d.M.mi_dpotrf_tiles if T.dtype == torch.float64 else d.M.mi_spotrf_tiles
    torch.cuda.synchronize()
    d.check(fn(d.h, N, NB, ctypes.c_void_p(T.data_ptr()), ctypes.byref(info)), "potrf")
    if info.value != 0:
        raise ValueError(f"matrix is not positive definite (info = {info.value})")


def _adjoint(T, G, N, NB):
    d = _Lib.get()
    fn = d.M.mi_dpotrf_adjoint_tiles if T.dtype == torch.float64 else d.M.mi_spotrf_adjoint_tiles
    torch.cuda.synchronize()
    d.check(fn(d.h, N, NB, ctypes.c_void_p(T.data_ptr()), ctypes.c_void_p(G.data_ptr())), "potrf adjoint")


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _ntiles(N, NB):
    MT = (N + NB - 1) // NB
    return MT * (MT + 1) // 2


# dplasmaUpper / dplasmaLower: the lower triangle of a row-major array is the
# upper triangle of the same memory read column-major
_UPPER, _LOWER = 121, 122
_STAGE_NB = 8160          # the staging kernels' largest tile


def _stage_in(A, N, NB):
    """Packed lower tiles of the lower triangle of the dense A (zero elsewhere)."""
    if A.shape != (N, N) or N == 0 or NB > _STAGE_NB:
        return to_tiles(A, NB)
    d = _Lib.get()
    A = A.resolve_neg().contiguous()
    T = A.new_empty((_ntiles(N, NB), NB, NB))
    fn = d.M.mi_dsym_lapack_to_tiles if A.dtype == torch.float64 else d.M.mi_ssym_lapack_to_tiles
    torch.cuda.synchronize()
    d.check(fn(d.h, _UPPER, N, _ptr(A), N, NB, _ptr(T)), "stage in")
    return T


def _stage_out(T, N, NB, symmetric):
    """The dense matrix of packed lower tiles: its lower triangle and zeros, or both triangles."""
    if N == 0 or NB > _STAGE_NB:
        A = from_tiles(T, N, NB)
        return A + A.tril(-1).T if symmetric else A
    d = _Lib.get()
    A = T.new_empty((N, N)) if symmetric else T.new_zeros((N, N))
    fn = d.M.mi_dsym_tiles_to_lapack if T.dtype == torch.float64 else d.M.mi_ssym_tiles_to_lapack
    torch.cuda.synchronize()
    d.check(fn(d.h, _UPPER, N, NB, _ptr(T), _ptr(A), N), "stage out")
    if symmetric:
        d.check(fn(d.h, _LOWER, N, NB, _ptr(T), _ptr(A), N), "stage out")
    return A


class Cholesky(torch.autograd.Function):
    """L = cholesky(A) (lower) on the tile kernels; backward on the adjoint kernels."""

    @staticmethod
    def forward(ctx, A, NB=512, recompute=False):
        if A.dtype not in (torch.float64, torch.float32) or A.device.type != "cuda":
            raise TypeError("Cholesky: A must be a float64 or float32 CUDA tensor")
        N = A.shape[0]
        T = _stage_in(A.detach(), N, NB)
        _potrf(T, N, NB)
        ctx.NB, ctx.N, ctx.recompute = NB, N, recompute
        ctx.save_for_backward(A.detach() if recompute else T)
        return _stage_out(T, N, NB, False)

    @staticmethod
    @once_differentiable
    def backward(ctx, gL):
        (saved,) = ctx.saved_tensors
        N, NB = ctx.N, ctx.NB
        if ctx.recompute:
            T = _stage_in(saved, N, NB)
            _potrf(T, N, NB)
        else:
            T = saved.contiguous()
        G = _stage_in(gL.to(T.dtype) if NB <= _STAGE_NB else gL.tril().to(T.dtype), N, NB)
        _adjoint(T, G, N, NB)
        return _stage_out(G, N, NB, True), None, None


class GpNll(torch.autograd.Function):
    """The likelihood of gp_nll as one pair of calls of the library, for data y
    that no gradient is wanted for."""

    @staticmethod
    def _forward(K, y, NB):
        d = _Lib.get()
        N = K.shape[0]
        K = K.resolve_neg().contiguous()
        T = K.new_empty((_ntiles(N, NB), NB, NB))
        a = y.resolve_neg().reshape(-1).clone(memory_format=torch.contiguous_format)
        out = torch.empty(2, dtype=torch.float64, device=K.device)
        info = ctypes.c_int(-1)
        fn = d.M.mi_dgp_nll if K.dtype == torch.float64 else d.M.mi_sgp_nll
        torch.cuda.synchronize()
        d.check(fn(d.h, N, NB, _ptr(K), N, _ptr(T), _ptr(a), _ptr(out), ctypes.byref(info)), "gp_nll")
        if info.value != 0:
            raise ValueError(f"matrix is not positive definite (info = {info.value})")
        return T, a, out

    @staticmethod
    def forward(ctx, K, y, NB, recompute):
        N = K.shape[0]
        T, a, out = GpNll._forward(K.detach(), y.detach(), NB)
        ctx.NB, ctx.N, ctx.recompute = NB, N, recompute
        ctx.save_for_backward(K.detach() if recompute else T, a)
        return (0.5 * out[1] + out[0] + 0.5 * N * math.log(2 * math.pi)).to(K.dtype)

    @staticmethod
    @once_differentiable
    def backward(ctx, g):
        d = _Lib.get()
        N, NB = ctx.N, ctx.NB
        T, a = (t.contiguous() for t in ctx.saved_tensors)
        if ctx.recompute:
            T = _stage_in(T, N, NB)
            _potrf(T, N, NB)
        alpha = torch.empty_like(a)
        G, dK = torch.empty_like(T), T.new_empty((N, N))
        scale = g.resolve_neg().reshape(1).contiguous()
        fn = d.M.mi_dgp_nll_grad if T.dtype == torch.float64 else d.M.mi_sgp_nll_grad
        torch.cuda.synchronize()
        d.check(fn(d.h, N, NB, _ptr(T), _ptr(a), _ptr(alpha), _ptr(scale), _ptr(G), _ptr(dK), N), "gp_nll gradient")
        return dK, None, None, None


def cholesky(A, NB=512, recompute=False):
    return Cholesky.apply(A, NB, recompute)


def se_kernel(X, lengthscale, variance=1.0, noise=1e-2):
    """Squared-exponential kernel v exp(-|x_i - x_j|^2 / (2 l^2)) + noise I."""
    d2 = (X * X).sum(1)[:, None] + (X * X).sum(1)[None, :] - 2.0 * X @ X.T
    d2 = d2.clamp_min(0.0)
    K = variance * torch.exp(-0.5 * d2 / lengthscale ** 2)
    return K + noise * torch.eye(X.shape[0], dtype=X.dtype, device=X.device)


def _whole_call(K, y, NB):
    """Whether gp_nll runs as GpNll: plain tensors that the library's calls
    take, and no derivative with respect to y (whose first and higher
    derivatives, backward or forward, go through torch's triangular solve).
    On an 8192-point FP64 problem that solve takes 9 of 33 ms, the copies
    between the dense and the tile layout by torch indexing another 5."""
    return (type(K) in (torch.Tensor, torch.nn.Parameter) and type(y) in (torch.Tensor, torch.nn.Parameter)
            and K.dtype in (torch.float64, torch.float32) and K.device.type == "cuda" and K.dim() == 2
            and K.shape[0] == K.shape[1] and K.shape[0] >= 1 and y.dtype == K.dtype and y.device == K.device
            and y.numel() == K.shape[0] and NB % 32 == 0 and 32 <= NB <= 960
            and not (y.requires_grad and torch.is_grad_enabled())
            and not torch._C._functorch.is_functorch_wrapped_tensor(K)
            and not torch._C._functorch.is_functorch_wrapped_tensor(y)
            and torch.autograd.forward_ad.unpack_dual(y).tangent is None
            and torch.autograd.forward_ad.unpack_dual(K).tangent is None)


def gp_nll(K, y, NB=512, recompute=False):
    """Negative log marginal likelihood of a Gaussian process:
    1/2 y^T K^-1 y + 1/2 logdet K + N/2 log 2 pi, with K = L L^T from the tile
    kernels: two triangular solves and logdet = 2 sum log diag(L)."""
    if _whole_call(K, y, NB):
        return GpNll.apply(K, y, NB, recompute)
    L = cholesky(K, NB, recompute)
    a = torch.linalg.solve_triangular(L, y.reshape(-1, 1), upper=False)
    return 0.5 * (a * a).sum() + torch.log(torch.diagonal(L)).sum() + 0.5 * y.numel() * math.log(2 * math.pi)
