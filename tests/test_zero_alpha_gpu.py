"""A device alpha of 0: B := 0 with A not referenced, on every path that tests alpha in its kernel
-- small, panel (16 and 32 vectors), chained (128- and 256-row super-blocks) -- and in time that
does not grow with one workgroup's share of a long triangle."""
import numpy as np
import pytest

import rocblas_amd as rb

pytestmark = pytest.mark.gpu
S = rb.rocblas_status
SHAPES = [(20, 9, 3), (33, 5, 1), (200, 40, 1), (200, 40, 300), (512, 100, 1), (513, 3, 1),
          (700, 40, 1), (1000, 300, 1), (2049, 260, 1)]


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("side", ["L", "R"])
def test_zero_alpha_on_the_device(side, prec):
    import torch
    from tests.gpu_util import GpuHandle
    h = GpuHandle()
    dt = torch.float64 if prec == "d" else torch.float32
    zero = torch.zeros(1, dtype=dt, device="cuda")
    rb.check(h.set_pointer_mode(rb.rocblas_pointer_mode.device))
    for k, nv, batch in SHAPES:
        print("zero alpha", side, prec, k, nv, batch, flush=True)
        m, n = (k, nv) if side == "L" else (nv, k)
        ld = m + 2
        B = torch.full((batch, n, ld), 3.0, dtype=dt, device="cuda")
        st = rb.trsm_strided_batched(h, side, "L", "N", "N", m, n, None, None, k, 0, B.data_ptr(),
                                     ld, ld * n, batch, precision=prec, alpha_ptr=zero.data_ptr())
        assert st == S.success
        out = B.cpu().numpy()
        assert not out[:, :, :m].any() and (out[:, :, m:] == 3.0).all()
    h.close()


def test_zeroing_a_long_solve_is_spread_over_workgroups():
    """16384 x 8, 1 MiB: far below the 140 us that one workgroup took (a launch takes 5)."""
    import torch
    from tests.gpu_util import GpuHandle
    h = GpuHandle()
    k, n = 16384, 8
    zero = torch.zeros(1, dtype=torch.float64, device="cuda")
    B = torch.full((n, k), 3.0, dtype=torch.float64, device="cuda")
    rb.check(h.set_pointer_mode(rb.rocblas_pointer_mode.device))
    call = lambda: rb.trsm(h, "L", "L", "N", "N", k, n, None, None, k, B.data_ptr(), k,
                           alpha_ptr=zero.data_ptr())
    best = 1e9
    for _ in range(5):
        t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        t0.record()
        for _ in range(20):
            assert call() == S.success
        t1.record()
        torch.cuda.synchronize()
        best = min(best, t0.elapsed_time(t1) / 20 * 1e3)
    assert not B.any()
    assert best < 50, best
    h.close()
