"""Triangular inverse and square at the edges of their levels and tiles.

Orders around the 16-column tiles, the diagonal block, two and three levels of
joined blocks (with a ragged or a missing last one), both triangles, with NaN
in the other triangle and the padding.  The inverse is checked as
||X L - I||_F <= 10 n eps cond, the square against the product in FP64 with the
inner-product bound 2 (n + 4) eps per entry of |L^H| |L|.
"""
import numpy as np
import pytest
import torch

from test_gpu_panel import TYPES, factor_of, spd, store

pytestmark = pytest.mark.gpu

ORDERS = [1, 15, 16, 17, 33, 64, 65, 127, 128, 129, 160, 255, 257, 384, 385, 512, 640, 1025]


def triangle(n, seed, dtype, uplo):
    L = torch.linalg.cholesky(spd(n, seed, dtype))
    L = L.to(dtype).to(L.dtype)
    return L if uplo == "L" else L.mH.contiguous()


def eps_of(prec):
    return np.finfo(np.float32 if prec in "SC" else np.float64).eps


@pytest.mark.parametrize("prec", "SDCZ")
@pytest.mark.parametrize("uplo", "LU")
@pytest.mark.parametrize("diag", "NU")
@pytest.mark.parametrize("n", ORDERS)
def test_trtri_levels(gpu, lapack, prec, uplo, diag, n):
    M = triangle(n, n + 3, TYPES[prec], uplo)
    if diag == "U":                      # a unit triangle with a moderate inverse; its diagonal is not read
        M = M / (2 * n)
        M.diagonal()[:] = 1.0
        M = M.to(TYPES[prec]).to(M.dtype)
    W = store(M, uplo, n + 1, TYPES[prec])
    if diag == "U":
        W[:, :n].diagonal()[:] = float("nan")
    st, info = getattr(gpu, f"cu{prec}trtri")(lapack, ord(uplo), ord(diag), n, gpu.ptr(W), n + 1)
    torch.cuda.synchronize()
    assert st == 0 and info == 0
    if diag == "U":
        assert torch.isnan(W[:, :n].diagonal()).all()
        W[:, :n].diagonal()[:] = 1.0
    X, L = factor_of(W, n, uplo), M if uplo == "L" else M.mH
    cond = (torch.linalg.norm(L) * torch.linalg.norm(X)).item()
    eye = torch.eye(n, device="cuda", dtype=X.dtype)
    assert torch.linalg.norm(X @ L - eye).item() <= 10 * n * eps_of(prec) * cond
    assert torch.isnan(W[:, n:]).all()


@pytest.mark.parametrize("prec", "SDCZ")
@pytest.mark.parametrize("uplo", "LU")
@pytest.mark.parametrize("n", ORDERS)
def test_lauum_edges(gpu, lapack, prec, uplo, n):
    M = triangle(n, n + 5, TYPES[prec], uplo)
    W = store(M, uplo, n + 1, TYPES[prec])
    st, info = getattr(gpu, f"cu{prec}lauum")(lapack, ord(uplo), n, gpu.ptr(W), n + 1)
    torch.cuda.synchronize()
    assert st == 0 and info == 0
    R = M.mH @ M if uplo == "L" else M @ M.mH
    bound = M.abs().mH @ M.abs() if uplo == "L" else M.abs() @ M.abs().mH
    got = factor_of(W, n, uplo)
    want = torch.tril(R if uplo == "L" else R.mH)
    low = torch.tril(bound if uplo == "L" else bound.mH)
    assert ((got - want).abs() <= 2 * (n + 4) * eps_of(prec) * low).all()
    if prec in "CZ":
        assert (got.diagonal().imag == 0).all()
    assert torch.isnan(W[:, n:]).all()


@pytest.mark.parametrize("prec", "SDCZ")
@pytest.mark.parametrize("uplo", "LU")
def test_potri_singular_is_untouched(gpu, lapack, prec, uplo):
    """A zero on the diagonal: info is its index and the matrix stays."""
    n, k = 300, 200
    M = triangle(n, 2, TYPES[prec], uplo)
    M[k, k] = 0.0
    W = store(M, uplo, n, TYPES[prec])
    before = W.clone()
    st, info = getattr(gpu, f"cu{prec}potri")(lapack, ord(uplo), n, gpu.ptr(W), n)
    torch.cuda.synchronize()
    assert st == 0 and info == k + 1
    assert torch.equal(torch.nan_to_num(W), torch.nan_to_num(before))


@pytest.mark.parametrize("uplo", "LU")
def test_trtri_large_tiles(gpu, lapack, uplo):
    """Levels that take the larger product tile, with a ragged last pair."""
    n = 6001
    M = triangle(n, n, torch.float64, uplo)
    W = store(M, uplo, n + 1, torch.float64)
    st, info = gpu.cuDtrtri(lapack, ord(uplo), gpu.NonUnit, n, gpu.ptr(W), n + 1)
    torch.cuda.synchronize()
    assert st == 0 and info == 0
    X, L = factor_of(W, n, uplo), M if uplo == "L" else M.mH
    cond = (torch.linalg.norm(L) * torch.linalg.norm(X)).item()
    eye = torch.eye(n, device="cuda", dtype=torch.float64)
    assert torch.linalg.norm(X @ L - eye).item() <= 10 * n * eps_of("D") * cond
    assert torch.isnan(W[:, n:]).all()


@pytest.mark.parametrize("uplo", "LU")
def test_potri_halved_square(gpu, lapack, uplo):
    """Above the order that is squared in one product: two halves and the
    products between them."""
    n = 8301
    A = spd(n, n, torch.float64)
    M = torch.linalg.cholesky(A)
    W = store(M if uplo == "L" else M.mH, uplo, n + 1, torch.float64)
    st, info = gpu.cuDpotri(lapack, ord(uplo), n, gpu.ptr(W), n + 1)
    torch.cuda.synchronize()
    assert st == 0 and info == 0
    X = factor_of(W, n, uplo)
    X = torch.tril(X) + torch.tril(X, -1).mT
    eye = torch.eye(n, device="cuda", dtype=torch.float64)
    err = (torch.linalg.norm(A @ X - eye) / (torch.linalg.norm(A) * torch.linalg.norm(X))).item()
    assert err <= 10 * n * eps_of("D"), err
    assert torch.isnan(W[:, n:]).all()
