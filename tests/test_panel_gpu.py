"""The panel solve (k <= 512 in one launch, panel_trsm.hpp) at the sizes where it can go wrong:
the edges of its 16-row sub-blocks, of the four wavefronts' shares and of its two register
layouts (k <= 256, k <= 512), vector counts around 16 and 32, one instance (16 vectors per
workgroup) and a batch wide enough for 32 vectors per workgroup, and diagonal blocks whose scaled
entries leave the floating-point range (the unscaled substitution)."""
import os
import re

import numpy as np
import pytest

import oracle
import rocblas_amd as rb
from rocblas_amd import build as rbuild

EPS = {"d": np.finfo(np.float64).eps, "s": np.finfo(np.float32).eps}


@pytest.fixture(scope="module")
def h():
    from tests.gpu_util import GpuHandle
    oracle.build()
    hd = GpuHandle()
    yield hd
    hd.close()


def run(h, side, uplo, trans, diag, m, n, alpha, A, B, batch, prec):
    """The batch (one triangle, `batch` copies of B) and the solution of one instance alone."""
    import torch
    from tests.gpu_util import gpu_trsm
    dt = np.float64 if prec == "d" else np.float32
    A, B = np.asfortranarray(A, dtype=dt), np.asfortranarray(B, dtype=dt)
    dA = torch.from_numpy(A.ravel(order="F").copy()).cuda()
    dB = torch.from_numpy(np.tile(B.ravel(order="F"), batch)).cuda()
    st = rb.trsm_strided_batched(h, side, uplo, trans, diag, m, n, alpha, dA.data_ptr(),
                                 A.shape[0], 0, dB.data_ptr(), B.shape[0], B.size, batch,
                                 precision=prec)
    assert st == rb.rocblas_status.success
    out = dB.cpu().numpy().reshape(batch, n, B.shape[0])
    assert (out == out[0]).all(), "instances differ"
    st, one = gpu_trsm(h, side, uplo, trans, diag, m, n, alpha, A, B, prec)
    assert st == rb.rocblas_status.success
    return out[0].T, one


CASES = [("L", "L", "N"), ("L", "U", "N"), ("L", "L", "T"), ("R", "U", "N"), ("R", "L", "T")]


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("k", [33, 49, 64, 65, 80, 113, 255, 256, 257, 272, 511, 512])
def test_edges_against_oracle_one_and_batched(h, k, prec):
    rng = np.random.default_rng(k)
    for i, (side, uplo, trans) in enumerate(CASES):
        nv = (1, 16, 17, 32, 33)[(i + k) % 5]
        batch = 520 if nv <= 16 else 260 if nv <= 32 else 175  # 512 vector groups or more
        m, n = (k, nv) if side == "L" else (nv, k)
        diag, alpha = "NU"[i % 2], (1.0, -0.5)[i % 2]
        print("panel", k, prec, side, uplo, trans, diag, nv, flush=True)
        A = oracle.diag_dominant_triangular(k, uplo, rng, lda=k + i)
        if diag == "U":
            oracle.make_unit_diagonal(A, uplo, k)
            A[np.arange(k), np.arange(k)] = np.nan
        A = np.asfortranarray(A.astype(np.float32 if prec == "s" else np.float64).astype(float))
        B = np.asfortranarray(rng.uniform(-1, 1, (m + 1, n)).astype(np.float32).astype(float))
        got, one = run(h, side, uplo, trans, diag, m, n, alpha, A, B, batch, prec)
        assert np.array_equal(got, one, equal_nan=True), "batched and single differ"
        assert np.array_equal(got[m:], B[m:]), "rows past m were written"
        ref = B.copy(order="F")
        oracle.trsm(side, uplo, trans, diag, m, n, alpha, A, ref)
        # the reference's bound on a solve's relative 1-norm error: 40 eps k
        X = np.asfortranarray(got[:m].astype(np.float64))
        assert oracle.norm1_rel_diff(m, n, X, ref[:m].copy(order="F")) <= 40 * EPS[prec] * k


@pytest.mark.gpu
@pytest.mark.parametrize("prec,big", [("d", 600), ("s", 70)])
def test_badly_scaled_triangles(h, prec, big):
    """Rows and columns scaled by powers of two up to 2^(+-big): entries divided by their column's
    diagonal overflow or vanish, though every step of the substitution is in range.  Scaling by
    powers of two commutes with rounding, so the solution is the plain one scaled, up to the
    rounding differences of two orders of evaluation (the bound of the unscaled problem)."""
    rng = np.random.default_rng(7)
    for k, n in ((64, 5), (100, 20), (300, 33)):
        print("badly scaled", prec, k, n, flush=True)
        dt = np.float32 if prec == "s" else np.float64
        A = oracle.diag_dominant_triangular(k, "L", rng).astype(dt).astype(np.float64)
        B = np.asfortranarray(rng.uniform(-1, 1, (k, n)).astype(dt).astype(np.float64))
        ref = B.copy(order="F")
        oracle.trsm("L", "L", "N", "N", k, n, 1.0, A, ref)
        # row scale r_i, column scale c_j: (R A C) (C^-1 X) = R B, every product r_i l_ij x_j in
        # range; r_i c_i (the diagonal) spreads over 2^(+-big)
        e = rng.integers(-big, big + 1, size=k)
        e[0], e[-1] = big, -big
        R, C = np.ldexp(1.0, e // 2), np.ldexp(1.0, e - e // 2)
        As = np.asfortranarray(np.tril(A) * R[:, None] * C[None, :])
        Bs = np.asfortranarray(B * R[:, None])
        assert np.isfinite(As.astype(dt)).all() and np.isfinite(Bs.astype(dt)).all()
        got, one = run(h, "L", "L", "N", "N", k, n, 1.0, As, Bs, 3, prec)
        assert np.array_equal(got, one)
        X = np.asfortranarray(got.astype(np.float64) * C[:, None])
        assert np.isfinite(X).all()
        assert oracle.norm1_rel_diff(k, n, X, ref) <= 40 * EPS[prec] * k


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["trsm", "trtri"])
def test_wait_timeout_is_reported_and_heals(op):
    """Waits inside a panel launch that give up (forced from the host: a few polls and an
    unreachable target, so every kernel still runs to its end): the next call of the handle reports
    it once and does no work, the one after that is right."""
    import torch
    from tests.gpu_util import GpuHandle
    rng = np.random.default_rng(9)
    k, nv = 200, 24
    A = np.nan_to_num(oracle.diag_dominant_triangular(k, "L", rng))
    dA = torch.from_numpy(A.ravel(order="F").copy()).cuda()
    B0 = torch.from_numpy(rng.uniform(-1, 1, k * (nv if op == "trsm" else k))).cuda()
    hd = GpuHandle()

    def call(B):
        if op == "trsm":
            st = rb.trsm(hd, "L", "L", "N", "N", k, nv, 1.0, dA.data_ptr(), k, B.data_ptr(), k)
        else:
            st = rb.trtri(hd, "L", "N", k, dA.data_ptr(), k, B.data_ptr(), k)
        torch.cuda.synchronize()
        return st, B

    S = rb.rocblas_status
    st, want = call(B0.clone())
    assert st == S.success
    assert hd.set_chain_test_timeout(1) == S.success
    print("panel timeout forced", op, flush=True)
    assert call(B0.clone())[0] == S.success
    assert hd.set_chain_test_timeout(0) == S.success
    st, B = call(B0.clone())
    assert st == S.internal_error and torch.equal(B, B0)
    print("panel after timeout", op, flush=True)
    st, B = call(B0.clone())
    assert st == S.success and torch.equal(B, want)
    assert hd.get_async_status() == S.success
    hd.close()


@pytest.mark.skipif(not os.path.exists(rbuild.HIPCC), reason="hipcc not available")
def test_every_panel_kernel_has_its_wait_states(tmp_path):
    """All kernels of panel_trsm.hip: no DPP hazard, no scratch."""
    from tests.test_dpp_hazards import compile_asm, kernels, scan
    asm = open(compile_asm(os.path.join(rbuild.CSRC, "panel_trsm.hip"), str(tmp_path / "p.s"))).read()
    found = {name: scan(body) for name, body in kernels(asm, r"panel_\w+kernel")}
    assert len(found) == 8, sorted(found)
    assert not any(found.values()), {k[:60]: v[:2] for k, v in found.items() if v}
    sizes = re.findall(r"\.amdhsa_private_segment_fixed_size (\d+)", asm)
    assert sizes and not any(int(x) for x in sizes), sizes
