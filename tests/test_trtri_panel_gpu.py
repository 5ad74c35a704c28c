"""Inverses built from panel-solved diagonal blocks (trtri_panel.hip): orders around the 16-row
panels, one block (up to 512), a short last block, batches; exact on a unit-diagonal integer
triangle and within the reference's trtri bound against the oracle."""
import os

import numpy as np
import pytest

import oracle
import rocblas_amd as rb
from rocblas_amd import build as rbuild


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("uplo", ["L", "U"])
def test_orders_around_the_panels(uplo, prec):
    import torch
    from tests.gpu_util import GpuHandle
    h = GpuHandle()
    rng = np.random.default_rng(5)
    dt = np.float64 if prec == "d" else np.float32
    for n, batch in ((33, 5), (47, 1), (48, 3), (255, 2), (256, 1), (257, 1), (511, 2), (512, 1),
                     (513, 1), (540, 1)):
        for diag in "NU":
            print("trtri panel", prec, uplo, diag, n, batch, flush=True)
            A = oracle.diag_dominant_triangular(n, uplo, rng, lda=n + 2)
            if diag == "U":
                oracle.make_unit_diagonal(A, uplo, n)
            A = A.astype(dt).astype(np.float64)
            ref = np.asfortranarray(np.nan_to_num(A[:n]))
            if diag == "U":
                ref[np.arange(n), np.arange(n)] = 1.0
            oracle.trtri(uplo, diag, n, ref)
            tri = np.tril(ref) if uplo == "L" else np.triu(ref)
            S = A.copy(order="F")
            if diag == "U":
                S[np.arange(n), np.arange(n)] = np.nan  # not read
            dA = torch.from_numpy(np.tile(S.ravel(order="F").astype(dt), batch)).cuda()
            dX = torch.full((batch * (n + 1) * n,), 7.0, dtype=dA.dtype, device="cuda")
            st = rb.trtri_strided_batched(h, uplo, diag, n, dA.data_ptr(), n + 2, (n + 2) * n,
                                          dX.data_ptr(), n + 1, (n + 1) * n, batch, precision=prec)
            assert st == rb.rocblas_status.success
            out = dX.cpu().numpy().reshape(batch, n, n + 1)
            assert (out == out[0]).all(), "instances differ"
            got = out[0].T
            assert (got[n] == 7.0).all(), "rows past n were written"
            opp = np.triu(got[:n], 1) if uplo == "L" else np.tril(got[:n], -1)
            assert not opp.any(), "opposite triangle"
            # clients/include/unit.hpp:631-638: eps * max(10000, n), relative
            err = np.abs(got[:n] - tri).max() / np.abs(tri).max()
            assert err <= np.finfo(dt).eps * max(10000, n), (n, err)
    # exact: ones on and below a unit diagonal have the bidiagonal inverse
    for n in (100, 300, 600):
        one = np.tril(np.ones((n, n))) if uplo == "L" else np.triu(np.ones((n, n)))
        dA = torch.from_numpy(np.asfortranarray(one).ravel(order="F").astype(dt)).cuda()
        dX = torch.empty_like(dA)
        assert rb.trtri(h, uplo, "U", n, dA.data_ptr(), n, dX.data_ptr(), n, precision=prec) == 0
        want = np.eye(n) - np.eye(n, k=-1 if uplo == "L" else 1)
        assert np.array_equal(dX.cpu().numpy().reshape(n, n).T, want.astype(dt)), n
    h.close()


@pytest.mark.skipif(not os.path.exists(rbuild.HIPCC), reason="hipcc not available")
def test_inverse_kernels_have_their_wait_states(tmp_path):
    from tests.test_dpp_hazards import compile_asm, kernels, scan
    asm = open(compile_asm(os.path.join(rbuild.CSRC, "trtri_panel.hip"), str(tmp_path / "t.s"))).read()
    found = {name: scan(body) for name, body in kernels(asm, "trtri_panel_kernel")}
    assert len(found) == 4, sorted(found)
    assert not any(found.values()), {k[:60]: v[:2] for k, v in found.items() if v}


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("uplo", ["L", "U"])
def test_two_pointer_arrays_of_the_same_matrices(uplo, prec):
    """In place through pointer arrays that differ: the host cannot see that some of their entries
    are equal.  Such an instance gives the bits of the same call out of place."""
    import torch
    from tests.gpu_util import GpuHandle
    h = GpuHandle()
    rng = np.random.default_rng(17)
    dt = np.float64 if prec == "d" else np.float32
    for n, batch in ((33, 7), (48, 3), (200, 5), (256, 2), (300, 3), (512, 2), (600, 3), (200, 300)):
        print("trtri in place, two arrays", prec, uplo, n, batch, flush=True)
        ld = n + 3
        A = oracle.diag_dominant_triangular(n, uplo, rng, lda=ld).astype(dt)
        dA = torch.from_numpy(np.tile(np.nan_to_num(A).ravel(order="F"), batch)).cuda()
        size = dA.element_size() * ld * n

        def call(a, x):
            pa = torch.tensor([a.data_ptr() + size * i for i in range(batch)]).cuda()
            # every third instance of an in-place call goes to a matrix of its own
            px = torch.tensor([(spare if i % 3 == 2 else x).data_ptr() + size * i
                               for i in range(batch)]).cuda()
            st = rb.trtri_batched(h, uplo, "N", n, pa.data_ptr(), ld, px.data_ptr(), ld, batch,
                                  precision=prec)
            assert st == rb.rocblas_status.success
            return [t.cpu().numpy().reshape(batch, n, ld)[:, :, :n] for t in (x, spare)]

        spare = torch.zeros_like(dA)
        want, wspare = call(dA, torch.zeros_like(dA))
        spare = torch.zeros_like(dA)
        got, gspare = call(dA, dA)
        for i in range(batch):
            w, g = (wspare[i], gspare[i]) if i % 3 == 2 else (want[i], got[i])
            assert np.array_equal(w, g), (n, i)
        tri = np.asfortranarray(np.nan_to_num(A[:n]).astype(np.float64))
        oracle.trtri(uplo, "N", n, tri)
        tri = np.tril(tri) if uplo == "L" else np.triu(tri)
        # clients/include/unit.hpp:631-638: eps * max(10000, n), relative
        assert np.abs(got[0].T - tri).max() / np.abs(tri).max() <= np.finfo(dt).eps * max(10000, n)
    h.close()


@pytest.mark.gpu
@pytest.mark.parametrize("uplo", ["L", "U"])
def test_strided_batches_that_meet_in_one_instance(uplo):
    """A at stride 2 S from 0, invA at stride S from S: the second instance's are the same memory."""
    import torch
    from tests.gpu_util import GpuHandle
    h = GpuHandle()
    rng = np.random.default_rng(23)
    for n in (40, 300, 600):
        print("trtri strided, one instance in place", uplo, n, flush=True)
        S = n * n
        mats = [np.nan_to_num(oracle.diag_dominant_triangular(n, uplo, rng)) for _ in range(2)]
        flat = [torch.from_numpy(M.ravel(order="F").copy()).cuda() for M in mats]
        buf = torch.zeros(3 * S, dtype=torch.float64, device="cuda")
        buf[:S], buf[2 * S:] = flat[0], flat[1]
        base = buf.data_ptr()
        assert rb.trtri_strided_batched(h, uplo, "N", n, base, n, 2 * S, base + 8 * S, n, S, 2) == 0
        for i in range(2):
            want = torch.zeros_like(flat[i])
            src = flat[i].repeat(2)  # as a batch: the same kernels
            out = want.repeat(2)
            assert rb.trtri_strided_batched(h, uplo, "N", n, src.data_ptr(), n, S, out.data_ptr(),
                                            n, S, 2) == 0
            assert torch.equal(buf[(i + 1) * S:(i + 2) * S], out[:S]), (n, i)
        assert torch.equal(buf[:S], flat[0])
    h.close()
