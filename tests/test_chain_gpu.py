"""The chained solve (chain_trsm.hip) at its edges: triangles just past the panel solve's 512 rows,
partial last super-blocks and sub-blocks, the register-narrow forms (up to 4, 8 and 16 vectors),
one and several panels, 128- and 256-row super-blocks, both storage orders and directions."""
import os

import numpy as np
import pytest

import oracle
import rocblas_amd as rb
from rocblas_amd import build as rbuild

EPS = {"d": np.finfo(np.float64).eps, "s": np.finfo(np.float32).eps}
SHAPES = [(513, 1), (528, 4), (600, 5), (640, 8), (700, 9), (769, 33), (1000, 40), (1025, 3),
          (1408, 130), (2049, 260)]  # the last two: more than 128 workgroups, then 256-row blocks


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("case", [("L", "L", "N"), ("L", "U", "N"), ("L", "L", "T"), ("L", "U", "T"),
                                  ("R", "L", "N"), ("R", "U", "T")])
def test_chain_edges_against_oracle(case, prec):
    from tests.gpu_util import GpuHandle, gpu_trsm
    side, uplo, trans = case
    h = GpuHandle()
    rng = np.random.default_rng(31)
    for i, (k, nv) in enumerate(SHAPES):
        m, n = (k, nv) if side == "L" else (nv, k)
        diag, alpha = "NU"[i % 2], (1.0, -0.5)[i % 2]
        print("chain", prec, case, diag, k, nv, flush=True)
        A = oracle.diag_dominant_triangular(k, uplo, rng, lda=k + i % 3)
        if diag == "U":
            oracle.make_unit_diagonal(A, uplo, k)
            A[np.arange(k), np.arange(k)] = np.nan
        dt = np.float64 if prec == "d" else np.float32
        A = np.asfortranarray(A.astype(dt))
        B = np.asfortranarray(rng.uniform(-1, 1, (m + i % 2, n)).astype(dt))
        st, got = gpu_trsm(h, side, uplo, trans, diag, m, n, alpha, A, B, prec)
        assert st == rb.rocblas_status.success
        st, again = gpu_trsm(h, side, uplo, trans, diag, m, n, alpha, A, B, prec)
        assert np.array_equal(got, again), "two runs differ"
        assert np.array_equal(got[m:], B[m:]), "rows past m were written"
        ref = np.asfortranarray(B.astype(np.float64))
        oracle.trsm(side, uplo, trans, diag, m, n, alpha, np.asfortranarray(A.astype(np.float64)),
                    ref)
        # the reference's bound on a solve's relative 1-norm error: 40 eps k
        X = np.asfortranarray(got[:m].astype(np.float64))
        assert oracle.norm1_rel_diff(m, n, X, ref[:m].copy(order="F")) <= 40 * EPS[prec] * k
    assert h.get_async_status() == rb.rocblas_status.success
    h.close()


@pytest.mark.skipif(not os.path.exists(rbuild.HIPCC), reason="hipcc not available")
def test_every_chain_kernel_has_its_wait_states(tmp_path):
    from tests.test_dpp_hazards import compile_asm, kernels, scan
    asm = open(compile_asm(os.path.join(rbuild.CSRC, "chain_trsm.hip"), str(tmp_path / "c.s"))).read()
    found = {name: scan(body) for name, body in kernels(asm, r"chain_\w+kernel")}
    assert len(found) == 8, sorted(found)
    assert not any(found.values()), {k[:60]: v[:2] for k, v in found.items() if v}
