"""The any-alignment GEMM (gemm_tile.hip), exact on small-integer data (every product and partial
sum is an integer below 2^24): its three tile sizes, 16- and 4-byte loads, each transpose form,
rows and columns around the tile edges, and K around whole steps (16 doubles, 32 floats)."""
import os
import re

import numpy as np
import pytest

import rocblas_amd as rb
from rocblas_amd import build as rbuild

# m, n, k, lda pad, ldb pad, ldc pad, alpha, beta, element shift of A and B
SHAPES = [
    (33, 64, 16, 0, 0, 0, 1.0, 0.0, 0),      # one 32 x 64 (FP64) / 64 x 64 (FP32) tile and a row
    (100, 130, 1, 1, 3, 0, -1.0, 1.0, 0),    # a single k
    (97, 131, 47, 1, 0, 2, -1.0, 1.0, 1),    # one short of three steps, everything odd
    (128, 192, 64, 0, 0, 0, -1.0, 1.0, 0),   # whole tiles and steps
    (64, 65, 33, 0, 5, 1, 1.0, 1.0, 0),
    (1028, 1060, 96, 0, 0, 0, -1.0, 1.0, 0), # 64 x 64 tiles, 16-byte loads, ragged edges
    (1025, 1027, 65, 1, 2, 0, -1.0, 1.0, 0), # 64 x 64 tiles, 4-byte loads, K one past a step
    (1090, 1100, 128, 1, 1, 1, 1.0, 0.0, 1),
    (2945, 2949, 32, 1, 1, 0, -1.0, 1.0, 0), # 128 x 128 tiles, 4-byte loads
    (2944, 3071, 64, 0, 0, 1, -1.0, 1.0, 1),
]


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("ops", ["NN", "TN", "NT", "TT"])
def test_tile_edges_exact(prec, ops):
    import torch
    from tests.gpu_util import GpuHandle
    h = GpuHandle()
    dt = torch.float64 if prec == "d" else torch.float32
    for m, n, k, pa, pb, pc, alpha, beta, shift in SHAPES:
        print("gemm tile", prec, ops, m, n, k, flush=True)
        gen = torch.Generator().manual_seed(m + n + k)
        mat = lambda r, c: torch.randint(-4, 5, (c, r), generator=gen, dtype=torch.int32).double()
        ar, ac = (m, k) if ops[0] == "N" else (k, m)
        br, bc = (k, n) if ops[1] == "N" else (n, k)
        A, B, C = mat(ar + pa, ac), mat(br + pb, bc), mat(m + pc, n)  # rows of these: columns
        opA = A[:, :ar].T if ops[0] == "N" else A[:, :ar]
        opB = B[:, :br].T if ops[1] == "N" else B[:, :br]
        want = C.clone()
        want[:, :m] = (alpha * (opA @ opB)).T + beta * C[:, :m]
        # NaN around the operands: nothing outside them may reach a result
        buf = lambda M: torch.cat([torch.full((shift,), np.nan, dtype=torch.float64), M.reshape(-1),
                                   torch.full((8,), np.nan, dtype=torch.float64)]).to(dt).cuda()
        A[:, ar:] = np.nan
        B[:, br:] = np.nan
        dA, dB, dC = buf(A), buf(B), C.to(dt).cuda()
        at = shift * dA.element_size()
        st = rb.gemm(h, ops[0], ops[1], m, n, k, alpha, dA.data_ptr() + at, ar + pa,
                     dB.data_ptr() + at, br + pb, beta, dC.data_ptr(), m + pc, precision=prec)
        assert st == rb.rocblas_status.success
        assert torch.equal(dC.cpu().double(), want), (m, n, k)
    h.close()


@pytest.mark.skipif(not os.path.exists(rbuild.HIPCC), reason="hipcc not available")
def test_tile_loads_are_set_up(tmp_path):
    """Every load into LDS follows the write of its destination to M0 and one wait state; no
    kernel spills."""
    from tests.test_dpp_hazards import compile_asm, kernels
    asm = open(compile_asm(os.path.join(rbuild.CSRC, "gemm_tile.hip"), str(tmp_path / "g.s"))).read()
    checked = 0
    for name, body in kernels(asm, "gemm_tile_kernel"):
        ops = [l.split(";")[0].strip() for _, l in body]
        ops = [o for o in ops if o and not o.startswith(".") and not o.endswith(":")]
        for i, o in enumerate(ops):
            if o.startswith("global_load_lds"):
                checked += 1
                assert ops[i - 1] == "s_nop 0", (name[:60], ops[i - 2:i + 1])
                m = re.match(r"s_mov_b32 m0, (\S+)$", ops[i - 2])
                assert m and not re.match(r"v\d|v\[", m.group(1)), (name[:60], ops[i - 2])
    assert checked > 0
    sizes = re.findall(r"\.amdhsa_private_segment_fixed_size (\d+)", asm)
    assert sizes and not any(int(x) for x in sizes), sizes
