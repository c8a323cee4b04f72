"""Diagonal block and panel solve of the factorisation at their edges.

Orders around the 4-column blocks of a leaf, the 16-column leaves, the
diagonal block (128 real, 64 complex) and, at n = 4300, the wider strips of the
panel solve; every precision and triangle, with NaN in the other triangle and
the padding rows (neither is read).  The bar is the backward error 10 n eps of
the precision, and the exact column of a failing pivot.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TYPES = {"S": torch.float32, "D": torch.float64, "C": torch.complex64, "Z": torch.complex128}


def spd(n, seed, dtype):
    g = torch.Generator(device="cuda").manual_seed(seed)
    wide = torch.complex128 if dtype.is_complex else torch.float64
    G = torch.randn(n, n, 2, generator=g, device="cuda", dtype=torch.float64)
    G = torch.view_as_complex(G) if dtype.is_complex else G[..., 0].contiguous()
    A = (G @ G.mH) / n
    A = torch.tril(A) + torch.tril(A, -1).mH
    A.diagonal().add_(0.5)
    return A.to(dtype).to(wide)          # exactly representable in dtype


def store(A, uplo, lda, dtype):
    """Column-major (n, lda) storage with NaN outside the triangle."""
    n = A.shape[0]
    W = torch.full((n, lda), float("nan"), device="cuda", dtype=dtype)
    keep = torch.ones(n, n, device="cuda", dtype=torch.bool)
    keep = torch.tril(keep) if uplo == "L" else torch.triu(keep)
    W[:, :n] = torch.where(keep, A, torch.full_like(A, float("nan"))).mT.to(dtype)
    return W


def factor_of(W, n, uplo):
    T = W[:, :n].mT.to(torch.complex128 if W.is_complex() else torch.float64)
    keep = torch.ones(n, n, device="cuda", dtype=torch.bool)
    keep = torch.tril(keep) if uplo == "L" else torch.triu(keep)
    T = torch.where(keep, T, torch.zeros_like(T))
    return T if uplo == "L" else T.mH


@pytest.mark.parametrize("prec", "SDCZ")
@pytest.mark.parametrize("uplo", "LU")
@pytest.mark.parametrize("n", [1, 3, 4, 5, 15, 16, 17, 20, 47, 63, 64, 65, 80, 111, 112, 113, 127, 129, 144, 193, 4300])
def test_potrf_edges(gpu, lapack, prec, uplo, n):
    if n == 4300 and prec in "CZ":
        pytest.skip("complex panels have one strip width")
    dtype = TYPES[prec]
    A = spd(n, 5 * n + 1, dtype)
    lda = n + 2
    W = store(A, uplo, lda, dtype)
    st, info = getattr(gpu, f"cu{prec}potrf")(lapack, ord(uplo), n, gpu.ptr(W), lda)
    torch.cuda.synchronize()
    assert st == 0 and info == 0
    L = factor_of(W, n, uplo)
    eps = np.finfo(np.float32 if prec in "SC" else np.float64).eps
    err = (torch.linalg.norm(A - L @ L.mH) / torch.linalg.norm(A)).item()
    assert err <= 10 * n * eps, err
    assert torch.isnan(W[:, n:]).all()
    if n > 1:
        other = torch.triu(torch.ones(n, n, device="cuda", dtype=torch.bool), 1)
        other = other if uplo == "L" else other.mT
        assert torch.isnan(W[:, :n].mT[other]).all()


@pytest.mark.parametrize("prec", "DZ")
@pytest.mark.parametrize("uplo", "LU")
@pytest.mark.parametrize("value", [-1.0, 0.0, float("nan")])
def test_potrf_failing_pivot(gpu, lapack, prec, uplo, value):
    """A pivot that becomes `value` after the elimination, in every column of
    two leaves and beyond the first diagonal block."""
    dtype, n = TYPES[prec], 150
    for k in list(range(0, 33)) + [63, 64, 100, 127, 128, 149]:
        L = torch.linalg.cholesky(spd(n, 9, dtype))
        L[k, k] = 0.0
        A = L @ L.mH
        A.diagonal()[k] += value if value != 0.0 else -1e-3   # rounding: an exact zero cannot be planted
        if value == 0.0 and k == 0:
            A.diagonal()[0] = 0.0
        W = store(A, uplo, n, dtype)
        st, info = getattr(gpu, f"cu{prec}potrf")(lapack, ord(uplo), n, gpu.ptr(W), n)
        assert st == 0 and info == k + 1, (k, info)


def imaginary_diagonal(n, value):
    g = torch.Generator(device="cuda").manual_seed(n)
    return 1.0 + 6.0 * torch.rand(n, generator=g, device="cuda", dtype=torch.float64) if value == "finite" \
        else torch.full((n,), float("nan"), device="cuda", dtype=torch.float64)


@pytest.mark.parametrize("prec", "CZ")
@pytest.mark.parametrize("uplo", "LU")
@pytest.mark.parametrize("n,value", [(n, "finite") for n in (1, 5, 16, 40, 64, 65, 150, 193)] +
                         [(n, "nan") for n in (1, 5, 16, 40, 64, 65, 150, 193, 700, 1100)])
def test_complex_diagonal_is_real(gpu, lapack, prec, uplo, n, value):
    """The imaginary part of the input's diagonal is not used: the factor and
    the inverse are those of the clean matrix to the bit, and their diagonals
    are real exactly."""
    dtype = TYPES[prec]
    clean = store(spd(n, 3 * n + 2, dtype), uplo, n + 1, dtype)
    dirty = clean.clone()
    k = torch.arange(n, device="cuda")
    torch.view_as_real(dirty)[k, k, 1] = imaginary_diagonal(n, value).to(torch.view_as_real(dirty).dtype)
    got = []
    for W in (clean, dirty):
        st, info = getattr(gpu, f"cu{prec}potrf")(lapack, ord(uplo), n, gpu.ptr(W), n + 1)
        assert st == 0 and info == 0
        F = factor_of(W, n, uplo).clone()
        st, info = getattr(gpu, f"cu{prec}potri")(lapack, ord(uplo), n, gpu.ptr(W), n + 1)
        assert st == 0 and info == 0
        X = factor_of(W, n, uplo).clone()
        assert (F.diagonal().imag == 0).all() and (X.diagonal().imag == 0).all()
        got.append((F, X))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("prec", "CZ")
@pytest.mark.parametrize("uplo", "LU")
@pytest.mark.parametrize("n,k", [(5, 3), (64, 40), (150, 64)])
def test_herk_ignores_imaginary_diagonal(gpu, blas, prec, uplo, n, k):
    """C's diagonal is real by definition: NaN in its imaginary part changes nothing."""
    dtype = TYPES[prec]
    A = torch.randn(k, n, device="cuda", dtype=dtype)
    clean = store(spd(n, n, dtype), uplo, n, dtype)
    dirty = clean.clone()
    i = torch.arange(n, device="cuda")
    torch.view_as_real(dirty)[i, i, 1] = float("nan")
    for W in (clean, dirty):
        st = getattr(gpu, f"cu{prec}herk")(blas, ord(uplo), gpu.NoTrans, n, k, -0.5, gpu.ptr(A), n, 0.75, gpu.ptr(W), n,
                                           torch.cuda.current_stream().cuda_stream)
        assert st == 0
    torch.cuda.synchronize()
    assert torch.equal(factor_of(clean, n, uplo), factor_of(dirty, n, uplo))
    assert (factor_of(dirty, n, uplo).diagonal().imag == 0).all()


@pytest.mark.parametrize("prec", "SD")
@pytest.mark.parametrize("uplo", "LU")
def test_potrf_long_panels(gpu, lapack, prec, uplo):
    """Panels with at least 8192 rows left apply the factored slices to each
    new one: the first two or three of this order."""
    dtype, n = TYPES[prec], 9293
    A = spd(n, n, dtype)
    lda = n + 3
    W = store(A, uplo, lda, dtype)
    st, info = getattr(gpu, f"cu{prec}potrf")(lapack, ord(uplo), n, gpu.ptr(W), lda)
    torch.cuda.synchronize()
    assert st == 0 and info == 0
    L = factor_of(W, n, uplo)
    eps = np.finfo(np.float32 if prec == "S" else np.float64).eps
    err = (torch.linalg.norm(A - L @ L.mT) / torch.linalg.norm(A)).item()
    assert err <= 10 * n * eps, err
    assert torch.isnan(W[:, n:]).all()
