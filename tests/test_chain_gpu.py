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
# 128-row super-blocks on 256 CUs: partial last blocks of 1, 16, 88, 0, 60, 1, 104 and 1 rows
SHAPES = [(513, 1), (528, 4), (600, 5), (640, 8), (700, 9), (769, 33), (1000, 40), (1025, 3),
          (1408, 130)]
# 256-row super-blocks: last blocks of 1, 5 16-row sub-blocks and 3 rows, 255 and 256 rows
LONG = [2049, 2048 + 16 * 5 + 3, 2048 + 255, 2304]


def long_shapes():
    """LONG with just enough vectors that 128-row blocks would be more workgroups than CUs (the
    rule of launch_chain), and still few enough for the chained solve (chain_fits)."""
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    out = []
    for k in LONG:
        panels, rows64 = cus // (-(-k // 128)) + 1, -(-k // 64)
        assert panels <= rows64 and rows64 * panels <= 8 * cus
        out.append((k, 16 * panels - 3))
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("case", [("L", "L", "N"), ("L", "U", "N"), ("L", "L", "T"), ("L", "U", "T"),
                                  ("R", "L", "N"), ("R", "U", "T")])
def test_chain_edges_against_oracle(case, prec):
    from tests.gpu_util import GpuHandle, gpu_trsm
    side, uplo, trans = case
    h = GpuHandle()
    rng = np.random.default_rng(31)
    for i, (k, nv) in enumerate(SHAPES + long_shapes()):
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
