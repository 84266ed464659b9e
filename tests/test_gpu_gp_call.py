"""gp_nll as one pair of library calls, and the staging of Cholesky, where they
can go wrong: ragged last tiles, a single element, an array that is not
contiguous, garbage above the diagonal, a scaled output gradient, recompute,
and data y that wants a gradient (which takes the general route).

K = B B^T / N + I has its eigenvalues in [1, 5.2] (B standard normal), so
solves, inverses and the reverse lose at most kappa^2 = 27 in the normwise
bound c N u kappa^2 on each of them; 64 N u of the largest entry (of the value,
for the likelihood) holds two or three such terms, with the FP64 formulas as
the reference."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ag(dp):
    import dplasma_amd.autograd as ag
    return ag


def problem(N, seed):
    rng = np.random.default_rng(seed)
    B = rng.standard_normal((N, N))
    K = B @ B.T / N + np.eye(N)
    return K, rng.standard_normal(N)


def reference(K, y):
    Ki = np.linalg.inv(K)
    al = Ki @ y
    nll = 0.5 * y @ al + 0.5 * np.linalg.slogdet(K)[1] + 0.5 * len(y) * np.log(2 * np.pi)
    return nll, 0.5 * (Ki - np.outer(al, al)), al


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("N,NB", [(1, 32), (31, 32), (96, 32), (129, 64), (333, 96), (513, 256), (700, 960)])
@pytest.mark.parametrize("how", ["plain", "strided", "recompute", "y_grad"])
def test_gp_call(ag, dtype, N, NB, how):
    K, y = problem(N, 100 + N)
    K = torch.tensor(K, dtype=dtype).double().numpy()        # as the device gets it
    y = torch.tensor(y, dtype=dtype).double().numpy()
    K = np.tril(K) + np.tril(K, -1).T
    nll, dK, al = reference(K, y)
    up = np.triu(np.full((N, N), np.nan), 1) if how == "plain" else 0.0
    Kt = torch.tensor(np.tril(K) + up if how == "plain" else K, dtype=dtype, device="cuda")
    if how == "strided":
        big = torch.zeros((N, 2 * N + 1), dtype=dtype, device="cuda")
        big[:, 1:2 * N + 1:2] = Kt
        Kt = big[:, 1:2 * N + 1:2]
        assert N == 1 or not Kt.is_contiguous()
    Kt.requires_grad_(True)
    yt = torch.tensor(y, dtype=dtype, device="cuda", requires_grad=how == "y_grad")
    out = ag.gp_nll(Kt, yt, NB, recompute=how == "recompute")
    assert out.dtype == dtype and out.dim() == 0
    assert ("GpNll" in type(out.grad_fn).__name__) == (how != "y_grad")
    (3.0 * out).backward()
    tol = 64 * max(N, 8) * torch.finfo(dtype).eps
    assert abs(float(out) - nll) <= tol * abs(nll)
    got = Kt.grad.double().cpu().numpy()
    assert np.abs(got - 3.0 * dK).max() <= tol * 3.0 * np.abs(dK).max()
    assert np.array_equal(got, got.T)
    if how == "y_grad":
        assert np.abs(yt.grad.double().cpu().numpy() - 3.0 * al).max() <= tol * 3.0 * np.abs(al).max()


def test_gp_call_refuses_an_indefinite_matrix(ag):
    K, y = problem(200, 7)
    K[150, 150] = -1.0
    with pytest.raises(ValueError, match="not positive definite"):
        ag.gp_nll(torch.tensor(K, device="cuda", requires_grad=True), torch.tensor(y, device="cuda"), 64)
