"""Host-side launch rules, compiled by themselves: launches of more workgroups than one launch can
have, which products run on the LDS-load tiles (CPU); solves and inverses that need several launches
(GPU)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import rocblas_amd as rb
from rocblas_amd import build as rbuild

CXX = shutil.which("g++")


def run_cpp(tmp_path, body, includes):
    src = tmp_path / "t.cpp"
    src.write_text("".join(f'#include "{i}"\n' for i in includes)
                   + "#include <cstdio>\nusing namespace rbamd;\nint main()\n{\n" + body + "}\n")
    exe = str(tmp_path / "t")
    subprocess.run([CXX, "-std=c++17", "-I", rbuild.CSRC, str(src), "-o", exe], check=True)
    return subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split()


@pytest.mark.skipif(CXX is None, reason="g++ not available")
@pytest.mark.parametrize("threads", [64, 256])
def test_slices_cover_every_workgroup_below_the_thread_limit(tmp_path, threads):
    sizes = [0, 1, 2**23 - 1, 2**23, 2**23 + 1, 2**24, 2**24 + 5, 2**31 - 1, 2**31, 2**32 + 7]
    body = "".join(f'for_launch_slices({n}ll, {threads}, [](long long f, unsigned c) '
                   f'{{ std::printf("%lld %u\\n", f, c); }}); std::puts("end -");\n' for n in sizes)
    out = run_cpp(tmp_path, body, ["launch_slices.hpp"])
    calls = iter(zip(out[::2], out[1::2]))
    for n in sizes:
        at = 0
        for first, count in calls:
            if first == "end":
                break
            assert int(first) == at and 0 < int(count) * threads < 2**32
            at += int(count)
        assert at == n


# (bytes per element, 16-byte loads, in a solve, A and B transposed, 64 x 64 tiles, K) of a product,
# and its measured time on the LDS-load tiles over the register-staged kernels' (256 CUs), where the
# two differ by 4% or more
MEASURED = [
    (4, 1, 0, 0, 0, 16, 256, 0.79), (4, 1, 0, 0, 0, 64, 64, 0.92), (4, 1, 1, 0, 0, 64, 256, 0.79),
    (4, 1, 0, 1, 0, 132, 320, 0.72), (4, 1, 0, 0, 0, 256, 1024, 0.49),
    (4, 0, 0, 0, 0, 63, 48, 1.55), (4, 0, 0, 0, 1, 16, 256, 1.41), (4, 0, 0, 0, 0, 64, 512, 1.44),
    (4, 0, 0, 0, 1, 64, 1024, 1.28), (4, 0, 0, 1, 0, 100, 320, 1.21), (4, 0, 0, 0, 1, 64, 4096, 0.82),
    (4, 0, 0, 0, 0, 128, 320, 1.40), (4, 0, 0, 1, 0, 128, 1024, 0.90), (4, 0, 0, 0, 0, 182, 64, 1.14),
    (4, 0, 0, 1, 0, 182, 1024, 0.83), (4, 0, 0, 0, 0, 256, 64, 0.93), (4, 0, 0, 1, 1, 1024, 256, 0.76),
    (4, 0, 1, 0, 0, 64, 320, 1.16), (4, 0, 1, 0, 0, 240, 384, 0.86), (4, 0, 1, 0, 0, 64, 1024, 0.92),
    (8, 1, 0, 0, 0, 16, 64, 0.86), (8, 1, 0, 0, 0, 64, 1024, 0.64), (8, 1, 0, 1, 0, 132, 64, 0.96),
    (8, 0, 0, 0, 0, 63, 48, 1.34), (8, 0, 0, 1, 0, 16, 256, 1.61), (8, 0, 1, 0, 0, 64, 320, 1.15),
    (8, 0, 0, 0, 1, 182, 4096, 1.14), (8, 0, 0, 0, 0, 165, 800, 1.12),
    (8, 0, 0, 0, 0, 256, 1024, 0.94), (8, 0, 0, 1, 0, 256, 1024, 1.05), (8, 0, 0, 0, 0, 506, 64, 0.94),
    (8, 0, 0, 1, 0, 1024, 256, 0.87)]


@pytest.mark.skipif(CXX is None, reason="g++ not available")
def test_products_run_on_the_kernel_that_measured_faster(tmp_path):
    body = "".join(f'std::printf("%d\\n", gemm_tile_pays({s}, {v}, {c}, {ta}, {tb}, {t}, {k}, 256));\n'
                   for s, v, c, ta, tb, t, k, _ in MEASURED)
    out = run_cpp(tmp_path, body, ["gemm_rule.hpp"])
    assert len(out) == len(MEASURED)
    for case, got in zip(MEASURED, out):
        assert int(got) == (case[-1] < 1), case


@pytest.mark.gpu
def test_more_workgroups_than_one_launch_can_have():
    """2^24 + 3 FP32 solves of order 33 with one triangle, as many solves of order 2 with one
    vector sixteen at a time (2^26 + 3: more than 2^32 threads), and the inverses of 5.6 million
    triangles of order 33 (three panels each): each in one call."""
    import torch
    from tests.gpu_util import GpuHandle
    h = GpuHandle()
    rng = np.random.default_rng(1)

    def triangle(k):
        A = np.tril(rng.uniform(-1, 1, (k, k))) / k + 1.5 * np.eye(k)
        return np.asfortranarray(A.astype(np.float32))

    # FP32 rounding of a well-conditioned triangle of this order: the reference's bound on a solve
    tol = lambda k: 40 * np.finfo(np.float32).eps * k
    for k, batch in ((33, 2**24 + 3), (2, 2**28 + 3)):
        print("many solves", k, batch, flush=True)
        A = triangle(k)
        dA = torch.from_numpy(A.ravel(order="F").copy()).cuda()
        b = rng.uniform(-1, 1, k).astype(np.float32)
        dB = torch.from_numpy(b).cuda().repeat(batch)
        st = rb.trsm_strided_batched(h, "L", "L", "N", "N", k, 1, 1.0, dA.data_ptr(), k, 0,
                                     dB.data_ptr(), k, k, batch, precision="s")
        assert st == rb.rocblas_status.success
        X = dB.view(batch, k)
        x = np.linalg.solve(A.astype(np.float64), b.astype(np.float64))
        assert np.abs(X[0].cpu().numpy() - x).max() <= tol(k) * np.abs(x).max()
        assert bool((X == X[0]).all()), "instances differ"
        del dB, X
    k, batch = 33, 2**24 // 3 + 5
    print("many inverses", k, batch, flush=True)
    A = triangle(k)
    dA = torch.from_numpy(A.ravel(order="F").copy()).cuda()
    dX = torch.full((batch * k * k,), 7.0, dtype=torch.float32, device="cuda")
    st = rb.trtri_strided_batched(h, "L", "N", k, dA.data_ptr(), k, 0, dX.data_ptr(), k, k * k,
                                  batch, precision="s")
    assert st == rb.rocblas_status.success
    X = dX.view(batch, k * k)
    inv = np.linalg.inv(A.astype(np.float64))
    assert np.abs(X[0].cpu().numpy().reshape(k, k).T - inv).max() <= tol(k) * np.abs(inv).max()
    assert bool((X == X[0]).all()), "instances differ"
    h.close()
