"""Infinities, NaN and zero pivots: they reach the rows that substitution reaches and no others.

The reference is plain substitution, x_j = c_j / L_jj and then c_i -= L_ij x_j for the rows below
only: which entries are finite has to agree exactly, finite ones within the reference's bound on a
solve's relative error (40 eps k).  Vectors without such values keep their bits whatever their
neighbours hold."""
import numpy as np
import pytest

import oracle
import rocblas_amd as rb

EPS = {"d": np.finfo(np.float64).eps, "s": np.finfo(np.float32).eps}
CASES = [("L", "L", "N"), ("L", "U", "N"), ("L", "L", "T"), ("R", "U", "N"), ("R", "L", "T")]


def substitution(M, C, first=None):
    """L^-1 C for a triangle M, lower or upper (then from the last row up); `first[v]`: row before
    which vector v is zero."""
    k = M.shape[0]
    upper = not np.tril(M, -1).any()
    L, x = (M[::-1, ::-1], C[::-1].copy()) if upper else (M, C.copy())
    with np.errstate(all="ignore"):
        for j in range(k):
            on = slice(None) if first is None else np.asarray(first) <= j
            x[j, on] /= L[j, j]
            x[j + 1:, on] -= L[j + 1:, j, None] * x[None, j, on]
    return x[::-1] if upper else x


@pytest.fixture(scope="module")
def h():
    from tests.gpu_util import GpuHandle
    oracle.build()
    hd = GpuHandle()
    yield hd
    hd.close()


def agree(got, want, k, prec):
    fin = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fin), "other entries are finite"
    g, w = np.where(fin, got, 0), np.where(fin, want, 0)
    scale = np.abs(w).sum(axis=0).max()
    assert np.abs(g - w).sum(axis=0).max() <= 40 * EPS[prec] * k * scale


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("k", [8, 20, 32, 33, 48, 64, 100, 200, 300, 512, 600])
def test_solves_with_infinities_and_zero_pivots(h, k, prec):
    from tests.gpu_util import gpu_trsm
    rng = np.random.default_rng(k)
    dt = np.float64 if prec == "d" else np.float32
    for i, (side, uplo, trans) in enumerate(CASES):
        for nv in (5, 20, 40):
            m, n = (k, nv) if side == "L" else (nv, k)
            print("nonfinite", k, prec, side, uplo, trans, nv, flush=True)
            A = oracle.diag_dominant_triangular(k, uplo, rng).astype(dt)
            A = np.nan_to_num(A)
            T = (np.tril if uplo == "L" else np.triu)(A).astype(np.float64)
            M = T if (trans == "N") == (side == "L") else T.T  # M X = B, or M X^T = B^T
            B = rng.uniform(-1, 1, (m, n)).astype(dt)
            vecs = (lambda X: X) if side == "L" else (lambda X: X.T)
            st, clean = gpu_trsm(h, side, uplo, trans, "N", m, n, 1.0, np.asfortranarray(A),
                                 np.asfortranarray(B), prec)
            assert st == rb.rocblas_status.success
            bad = B.copy()
            for v, (row, value) in enumerate([(k // 2, np.inf), (5, -np.inf), (k - 1, np.nan),
                                              (k - 3, np.inf)]):
                vecs(bad)[row, v] = value
            st, got = gpu_trsm(h, side, uplo, trans, "N", m, n, 1.0, np.asfortranarray(A),
                               np.asfortranarray(bad), prec)
            assert st == rb.rocblas_status.success
            agree(vecs(got), substitution(M, vecs(bad).astype(np.float64)), k, prec)
            assert np.array_equal(vecs(got)[:, 4:], vecs(clean)[:, 4:]), "finite vectors changed"
            # a zero pivot
            S, j = A.copy(), (k // 2, 7, k - 1, 0, k - 2)[i]
            S[j, j] = 0.0
            M = M.copy()
            M[j, j] = 0.0
            st, got = gpu_trsm(h, side, uplo, trans, "N", m, n, 1.0, np.asfortranarray(S),
                               np.asfortranarray(B), prec)
            assert st == rb.rocblas_status.success
            agree(vecs(got), substitution(M, vecs(B).astype(np.float64)), k, prec)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("uplo", ["L", "U"])
def test_inverses_with_zero_pivots(h, uplo, prec):
    """Columns past a zero pivot are those of the regular triangle below it; the opposite triangle
    stays zero.  (One diagonal block of the blocked inverse: up to 512 rows.)"""
    import torch
    rng = np.random.default_rng(3)
    dt = np.float64 if prec == "d" else np.float32
    for n, j in ((33, 0), (40, 5), (48, 31), (64, 63), (100, 40), (256, 128), (300, 17), (512, 500)):
        print("singular inverse", uplo, prec, n, j, flush=True)
        A = np.nan_to_num(oracle.diag_dominant_triangular(n, uplo, rng)).astype(dt)
        A = (np.tril if uplo == "L" else np.triu)(A)
        A[j, j] = 0.0
        dA = torch.from_numpy(A.ravel(order="F").copy()).cuda()
        dX = torch.full_like(dA, 3.0)
        assert rb.trtri(h, uplo, "N", n, dA.data_ptr(), n, dX.data_ptr(), n, precision=prec) == 0
        got = dX.cpu().numpy().reshape(n, n).T
        first = np.arange(n) if uplo == "L" else np.arange(n)[::-1]
        agree(got, substitution(A.astype(np.float64), np.eye(n), first), n, prec)
        opp = np.triu(got, 1) if uplo == "L" else np.tril(got, -1)
        assert not opp.any(), "opposite triangle"
