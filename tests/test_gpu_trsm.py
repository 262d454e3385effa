"""GPU: the one-launch triangular solves (up to 256 rows, 32 at a time) against LAPACK, at
the sizes around their steps and tiles: one step, partial steps (panel widths that are not
multiples of 32), one launch's most rows and one step past it, columns that fill part of a
16-column workgroup.

Tolerance: a backward-stable solve has |A x - b| <= c n u (|L||U| |x|) with c of a few; 8
is used, and LAPACK's own residual on these inputs is about 0.1 of that bound."""
import numpy as np
import pytest
import scipy.linalg
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [32, 96, 256, 288, 544])
@pytest.mark.parametrize("nrhs", [1, 17, 70])
def test_batched_solve(ctx, n, nrhs):
    rng = np.random.default_rng(n + nrhs)
    nbat = 2
    A = rng.standard_normal((nbat, n, n))
    B = rng.standard_normal((nbat, n, nrhs))
    LU, perm = np.empty_like(A), np.empty((nbat, n), dtype=np.int32)
    for z in range(nbat):
        LU[z], piv = scipy.linalg.lu_factor(A[z])
        p = np.arange(n)
        for i, q in enumerate(piv):
            p[[i, q]] = p[[q, i]]
        perm[z] = p
    dLU = torch.tensor(np.ascontiguousarray(LU.transpose(0, 2, 1)), device="cuda").transpose(1, 2)
    dB = torch.tensor(np.ascontiguousarray(B.transpose(0, 2, 1)), device="cuda").transpose(1, 2)
    X = ctx.lu_solve_batched(dLU, torch.tensor(perm, device="cuda"), dB).cpu().numpy()
    for z in range(nbat):
        L, U = np.tril(LU[z], -1) + np.eye(n), np.triu(LU[z])
        bound = 8 * n * 2.0 ** -53 * (np.abs(L) @ (np.abs(U) @ np.abs(X[z])))
        assert (np.abs((L @ (U @ X[z]))[np.argsort(perm[z])] - B[z]) <= bound[np.argsort(perm[z])]).all()


@pytest.mark.parametrize("prec,u", [("f64", 2.0 ** -53), ("f32", 2.0 ** -24)])
@pytest.mark.parametrize("n,nb", [(300, 48), (301, 112), (700, 208), (1100, 512)])
def test_factor_with_any_panel_width(ctx, prec, u, n, nb):
    dt = np.float64 if prec == "f64" else np.float32
    A = np.random.default_rng(n).standard_normal((n, n)).astype(dt)
    dA = torch.tensor(np.ascontiguousarray(A.T), device="cuda").T
    ipiv, perm, info = ctx.lu_factor(prec, dA, nb)
    F, p = dA.cpu().numpy().astype(np.float64), perm.cpu().numpy()
    assert info == 0
    L, U = np.tril(F, -1) + np.eye(n), np.triu(F)
    err = np.abs(L @ U - A.astype(np.float64)[p])
    assert (err <= 8 * n * u * (np.abs(L) @ np.abs(U))).all(), (err / (np.abs(L) @ np.abs(U))).max() / (n * u)


@pytest.mark.filterwarnings("ignore::scipy.linalg.LinAlgWarning")
@pytest.mark.parametrize("prec,u", [("f64", 2.0 ** -53), ("f32", 2.0 ** -24)])
@pytest.mark.parametrize("n", [1, 31, 33, 37, 255, 1023, 1024, 1025, 1100, 1281])
def test_panel_shapes(ctx, prec, u, n):
    """One row per thread: a panel of one workgroup (up to 1024 rows) and of several, rows
    that fill part of the last one, panels narrower than 32 columns and not a multiple of
    the 4 columns between two rotations.  The pivots are LAPACK's where no two candidates are
    within rounding (normal entries: all of them in fp64, the first panel's in fp32); integer
    entries tie in the first column."""
    dt = np.float64 if prec == "f64" else np.float32
    rng = np.random.default_rng(n)
    A = rng.integers(-3, 4, (n, n)).astype(dt) if n % 2 else rng.standard_normal((n, n)).astype(dt)
    dA = torch.tensor(np.ascontiguousarray(A.T), device="cuda").T
    ipiv, perm, info = ctx.lu_factor(prec, dA)
    F, p, piv = dA.cpu().numpy().astype(np.float64), perm.cpu().numpy(), ipiv.cpu().numpy()
    assert (piv >= np.arange(n)).all() and (piv < n).all()
    assert int(piv[0]) == int(np.argmax(np.abs(A[:, 0])))
    ref, rpiv = scipy.linalg.lu_factor(A)
    zeros = np.flatnonzero(np.diag(ref) == 0)  # (of these inputs, n = 1 is the matrix 0)
    assert info == (zeros[0] + 1 if zeros.size else 0) and (info == 0 or n == 1)
    if n % 2 == 0:
        k = n if prec == "f64" else 32
        assert piv[:k].tolist() == rpiv[:k].tolist()
    L, U = np.tril(F, -1) + np.eye(n), np.triu(F)
    assert np.abs(L).max() <= 1.0
    err = np.abs(L @ U - A.astype(np.float64)[p])
    assert (err <= 8 * n * u * (np.abs(L) @ np.abs(U)) + 1e-300).all()
