"""Residuals on graded factors: squared-exponential covariances.

The Cholesky factor of exp(-(x - y)^2 / (2 l^2)) + nugget I on a grid has
columns that fall by orders of magnitude, so that a product with the inverse of
a block loses digits where a substitution does not; matrices of independent
entries do not show it.  The bars are 10 n eps times the norms of the factors of
the residual, with no condition number: a row-by-row substitution meets them
with two digits to spare.
"""
from decimal import Decimal, localcontext
from fractions import Fraction

import numpy as np
import pytest
import torch

from test_gpu_panel import TYPES, factor_of, store

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def covariance(n, length, nugget, dtype):
    x = torch.linspace(0.0, 1.0, n, device="cuda", dtype=torch.float64)
    A = torch.exp(-((x[:, None] - x) ** 2) / (2.0 * length * length)) + nugget * torch.eye(n, device="cuda", dtype=torch.float64)
    if not dtype.is_complex:
        return A
    k = torch.arange(n, device="cuda", dtype=torch.float64)
    p = torch.polar(torch.ones_like(k), 0.37 * k * k)        # D A D^H: the same grading, complex entries
    A = p[:, None] * A * p.conj()
    A = torch.tril(A) + torch.tril(A, -1).mH
    A.diagonal().imag.zero_()
    return A


def norm(M):
    return torch.linalg.norm(M).item()


def lower_factor(n, length, nugget, dtype):
    return torch.linalg.cholesky(covariance(n, length, nugget, dtype))


@pytest.mark.parametrize("prec", "DZ")
@pytest.mark.parametrize("uplo", "LU")
@pytest.mark.parametrize("n", [20, 60, 64, 100, 128])
def test_trsm_residual(gpu, blas, prec, uplo, n):
    """L X = B, from L and from U = L^H: the sides that a substitution solves
    with a residual free of the condition number."""
    dtype = TYPES[prec]
    L = lower_factor(n, 0.05, 1e-10, dtype)
    W = store(L if uplo == "L" else L.mH, uplo, n + 1, dtype)
    g = torch.Generator(device="cuda").manual_seed(n)
    B = torch.randn(20, n, 2, generator=g, device="cuda", dtype=torch.float64)
    B = torch.view_as_complex(B) if dtype.is_complex else B[..., 0].contiguous()
    X = B.clone()
    trans = gpu.NoTrans if uplo == "L" else (gpu.ConjTrans if dtype.is_complex else gpu.Trans)
    st = getattr(gpu, f"cu{prec}trsm")(blas, gpu.Left, ord(uplo), trans, gpu.NonUnit, n, 20, 1.0, gpu.ptr(W), n + 1,
                                       gpu.ptr(X), n, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert st == 0
    err = norm(L @ X.mT - B.mT) / (norm(L) * norm(X) + norm(B))
    assert err <= 10 * n * EPS, err


@pytest.mark.parametrize("uplo", "LU")
@pytest.mark.parametrize("prec,n", [(p, n) for p in "DZ" for n in (20, 48, 60, 64, 100, 128) if p == "D" or n <= 64])
def test_trtri_residual(gpu, lapack, prec, uplo, n):
    """||L X - I|| of one diagonal block (up to 64 complex, 128 real)."""
    L = lower_factor(n, 0.05, 1e-10, TYPES[prec])
    W = store(L if uplo == "L" else L.mH, uplo, n + 1, TYPES[prec])
    st, info = getattr(gpu, f"cu{prec}trtri")(lapack, ord(uplo), gpu.NonUnit, n, gpu.ptr(W), n + 1)
    torch.cuda.synchronize()
    assert st == 0 and info == 0
    X = factor_of(W, n, uplo)
    err = norm(L @ X - torch.eye(n, device="cuda", dtype=X.dtype)) / (norm(L) * norm(X))
    assert err <= 10 * n * EPS, err


@pytest.mark.parametrize("uplo", "LU")
@pytest.mark.parametrize("n,length,nugget", [(60, 0.05, 1e-8), (128, 0.05, 1e-8), (512, 0.05, 1e-10)])
def test_potrs_residual(gpu, lapack, uplo, n, length, nugget):
    A = covariance(n, length, nugget, torch.float64)
    W = store(A, uplo, n + 1, torch.float64)
    g = torch.Generator(device="cuda").manual_seed(n)
    B = torch.randn(20, n, generator=g, device="cuda", dtype=torch.float64)
    X = B.clone()
    st, info = gpu.cuDpotrf(lapack, ord(uplo), n, gpu.ptr(W), n + 1)
    assert st == 0 and info == 0
    st, info = gpu.cuDpotrs(lapack, ord(uplo), n, 20, gpu.ptr(W), n + 1, gpu.ptr(X), n)
    torch.cuda.synchronize()
    assert st == 0 and info == 0
    err = norm(A @ X.mT - B.mT) / (norm(A) * norm(X) + norm(B))
    assert err <= 10 * n * EPS, err


@pytest.mark.parametrize("uplo", "LU")
@pytest.mark.parametrize("n", [60, 100, 128])
def test_potri_residual(gpu, lapack, uplo, n):
    A = covariance(n, 0.1, 1e-8, torch.float64)
    W = store(A, uplo, n + 1, torch.float64)
    st, info = gpu.cuDpotrf(lapack, ord(uplo), n, gpu.ptr(W), n + 1)
    assert st == 0 and info == 0
    st, info = gpu.cuDpotri(lapack, ord(uplo), n, gpu.ptr(W), n + 1)
    torch.cuda.synchronize()
    assert st == 0 and info == 0
    X = factor_of(W, n, uplo)
    X = torch.tril(X) + torch.tril(X, -1).mH
    err = norm(A @ X - torch.eye(n, device="cuda", dtype=X.dtype)) / (norm(A) * norm(X))
    assert err <= 10 * n * EPS, err


@pytest.mark.parametrize("uplo", "LU")
def test_batched_inverse_residual(gpu, lapack, uplo):
    """The three size classes of the batched plan, at their edges."""
    cases = [(16, 0.1), (17, 0.1), (60, 0.1), (64, 0.1), (65, 0.1), (100, 0.1), (128, 0.1), (129, 0.05), (250, 0.02),
             (256, 0.02)]
    mats = [covariance(n, length, 1e-8, torch.float64) for n, length in cases]
    sizes = [n for n, _ in cases]
    offs = [int(v) for v in np.cumsum([0] + [n * n for n in sizes[:-1]])]
    W = torch.cat([M.reshape(-1) for M in mats])
    logdet = torch.zeros(len(sizes), device="cuda", dtype=torch.float64)
    info = torch.full((len(sizes),), -9, device="cuda", dtype=torch.int32)
    with gpu.BatchedPlan(lapack, ord(uplo), "D", sizes, offs) as plan:
        assert plan.status == 0
        assert plan.run_inverse(gpu.ptr(W), gpu.ptr(logdet), gpu.ptr(info), torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
    assert (info == 0).all()
    for n, o, A in zip(sizes, offs, mats):
        X = factor_of(W[o:o + n * n].reshape(n, n), n, uplo)
        X = torch.tril(X) + torch.tril(X, -1).mT
        err = norm(A @ X - torch.eye(n, device="cuda", dtype=X.dtype)) / (norm(A) * norm(X))
        assert err <= 10 * n * EPS, (n, err)


def exact_logdet(M):
    """Pivots in rational arithmetic, their logarithms with 50 digits."""
    n = len(M)
    F = [[Fraction(float(v)) for v in row] for row in M]
    with localcontext() as ctx:
        ctx.prec = 50
        total = Decimal(0)
        for k in range(n):
            total += Decimal(F[k][k].numerator).ln() - Decimal(F[k][k].denominator).ln()
            for i in range(k + 1, n):
                f = F[i][k] / F[k][k]
                for j in range(k, n):
                    F[i][j] -= f * F[k][j]
        return float(total)


@pytest.mark.parametrize("n", [2, 3, 5])
def test_small_logdet_is_exact_to_the_condition(gpu, lapack, n):
    """Log-determinants of ill-conditioned small matrices from the batched plan
    and from the task-graph plan against exact arithmetic.  L L^T = A + E with
    ||E|| <= (n + 1) eps n ||A|| moves the log-determinant by at most sqrt(n)
    ||E|| / s_min, the n logarithms and their sum by 10 n eps relative."""
    count = 150
    rng = np.random.default_rng(n)
    G = rng.standard_normal((count, n, n))
    A = G @ np.swapaxes(G, 1, 2) / n + np.exp(rng.uniform(np.log(1e-8), 0.0, count))[:, None, None] * np.eye(n)
    A = np.tril(A) + np.swapaxes(np.tril(A, -1), 1, 2)
    want = np.array([exact_logdet(M) for M in A])
    bound = (n ** 1.5 * (n + 1) * np.linalg.cond(A) + 10 * n * np.maximum(1.0, np.abs(want))) * EPS
    sizes, offs, offb = [n] * count, [i * n * n for i in range(count)], [i * n for i in range(count)]
    W = torch.from_numpy(A.reshape(-1).copy()).cuda()
    A0 = W.clone()
    logdet = torch.zeros(2, count, device="cuda", dtype=torch.float64)
    info = torch.zeros(count, device="cuda", dtype=torch.int32)
    with gpu.BatchedPlan(lapack, gpu.Lower, "D", sizes, offs) as plan:
        assert plan.run(gpu.ptr(W), gpu.ptr(logdet[0]), gpu.ptr(info), torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
    assert (info == 0).all()
    B = torch.ones(count * n, device="cuda", dtype=torch.float64)
    X, Ainv, iters = torch.zeros_like(B), torch.zeros_like(A0), torch.zeros_like(info)
    with gpu.BatchedSolvePlan(lapack, gpu.Lower, sizes, offs, 1, offb) as plan:
        assert plan.run(gpu.ptr(A0), gpu.ptr(B), gpu.ptr(X), gpu.ptr(Ainv), gpu.ptr(iters), gpu.ptr(logdet[1]),
                        gpu.ptr(info)) == 0
        torch.cuda.synchronize()
    assert (info == 0).all()
    for got in logdet.cpu().numpy():
        assert np.all(np.abs(got - want) <= bound)
