"""Performance cases of the triangular-solve library, each one pass through a public entry point.

What is covered: ``trsm`` as a single call, as a strided batch and as a batch of pointer arrays, the
variable-size batch (``trsm_vbatched``) and ``trtri``, in FP64 and FP32, over sides, triangles,
transposes and diagonals, from one tiny solve to 16384 x 16384.  Matrices are column-major with the
leading dimension ``rows + pad``; operands live in device memory and are solved in place, as a
factorisation or a solver that calls this library does.

Inputs: the triangle's diagonal is U[1, 2] and its other entries U[-1, 1] / k (well conditioned; the
same distribution as ``rocblas_amd.synth.tri_uniform``), the other triangle holds U[-1, 1] values that
no call may read, and the right-hand sides are U[-1, 1].

``listed()`` names the cases, ``draw(rng)`` gives one more of the same ranges, ``prepare(case, seed)``
builds what a caller holds before the call, ``run(state)`` is the call, ``work(case)`` the bytes and
operations it cannot do without, and ``exact(case, seed)`` its result in 64 bits by plain torch.
"""
import math
import random

import torch

import rocblas_amd as rb


def _trsm(name, prec, side, uplo, trans, diag, m, n, form="single", batch=1, pad=0, alpha=1.0):
    return {"name": name, "op": "trsm", "prec": prec, "side": side, "uplo": uplo, "trans": trans,
            "diag": diag, "m": m, "n": n, "form": form, "batch": batch, "pad": pad, "alpha": alpha}


def listed():
    return [
        # one tiny solve: a Kalman filter's or a block preconditioner's single call, all launch
        # latency and host path
        _trsm("single_32x8", "d", "L", "L", "N", "N", 32, 8),
        # thousands of order-32 solves at once: block-Jacobi preconditioners, batched Cholesky
        # solves of small systems
        _trsm("batch_32x16_x20000", "d", "L", "L", "N", "N", 32, 16, "strided", 20000),
        # the transposed second half of such a solve with vectors in rows, FP32, odd sizes
        _trsm("batch_f32_50x23_x10000", "s", "R", "U", "T", "N", 50, 23, "strided", 10000),
        # blocks of a batched factorisation given as pointer arrays, order a few hundred
        _trsm("batch_200x64_x256", "d", "L", "L", "N", "N", 200, 64, "pointers", 256),
        # one mid-size solve whose latency a caller waits for
        _trsm("single_512x256", "d", "L", "L", "N", "N", 512, 256),
        # a long triangle with few right-hand sides: back substitution after a factorisation
        _trsm("single_4096x8", "d", "L", "U", "N", "N", 4096, 8),
        # the panel update of a blocked Cholesky factorisation, X L^T = A21, ragged row count
        _trsm("cholesky_panel_6001x512", "d", "R", "L", "T", "N", 6001, 512),
        # the block row of an LU factorisation, unit lower triangle
        _trsm("lu_row_2048x2048", "d", "L", "L", "N", "U", 2048, 2048),
        # an FP32 system of odd order, odd leading dimensions
        _trsm("square_f32_3001x2999", "s", "L", "L", "T", "N", 3001, 2999),
        # the largest blocked solve
        _trsm("square_16384", "d", "L", "U", "N", "N", 16384, 16384),
        # instances of many sizes in one call: fronts of a sparse factorisation
        {"name": "vbatch_8_512_x4096", "op": "vbatched", "prec": "d", "side": "L", "uplo": "L",
         "trans": "N", "diag": "N", "lo": 8, "hi": 512, "nhi": 64, "batch": 4096, "sizes": 0},
        # explicit inverse of a Cholesky factor (covariances, preconditioners)
        {"name": "trtri_3000", "op": "trtri", "prec": "d", "uplo": "L", "diag": "N", "n": 3000,
         "batch": 1, "pad": 0},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    prec = rng.choice("dds")
    side, uplo, trans = rng.choice("LR"), rng.choice("LU"), rng.choice("NT")
    diag = rng.choice("NNNU")
    pad = rng.choice((0, 0, 0, 1, 5, 32))
    alpha = rng.choice((1.0, 1.0, -1.0, 0.75))
    family = rng.random()
    if family < 0.45:  # one solve
        k, v = _log_int(rng, 16, 8192), _log_int(rng, 1, 8192)
        m, n = (k, v) if side == "L" else (v, k)
        c = _trsm("", prec, side, uplo, trans, diag, m, n, "single", 1, pad, alpha)
    elif family < 0.75:  # a batch of equal sizes
        k, v = _log_int(rng, 4, 512), _log_int(rng, 1, 256)
        m, n = (k, v) if side == "L" else (v, k)
        most = max(1, 150_000_000 // ((k + pad) * k + (m + pad) * n))
        batch = min(_log_int(rng, 16, 20000), most)
        c = _trsm("", prec, side, uplo, trans, diag, m, n, rng.choice(("strided", "pointers")),
                  batch, pad, alpha)
    elif family < 0.85:  # instances of many sizes
        hi = _log_int(rng, 64, 512)
        c = {"op": "vbatched", "prec": prec, "side": side, "uplo": uplo, "trans": trans,
             "diag": diag, "lo": 8, "hi": hi, "nhi": _log_int(rng, 4, 64),
             "batch": _log_int(rng, 256, 4096), "sizes": rng.randrange(1 << 20)}
    else:  # inverses
        n = _log_int(rng, 16, 6000)
        batch = 1 if n > 256 else rng.choice((1, _log_int(rng, 16, 4000)))
        c = {"op": "trtri", "prec": prec, "uplo": uplo, "diag": diag, "n": n, "batch": batch,
             "pad": pad}
    c.pop("name", None)
    return c


def _dtype(case):
    return torch.float64 if case["prec"] == "d" else torch.float32


def _uniform(gen, count, dtype):
    """U[-1, 1] values on the device, from the generator."""
    return torch.rand(count, generator=gen, dtype=dtype, device="cuda").mul_(2.0).sub_(1.0)


def _triangles(gen, k, ld, batch, dtype):
    """batch k x k matrices, column-major with leading dimension ld (rows past k hold U[-1, 1] too):
    a flat tensor in which column j of matrix b starts at (b k + j) ld."""
    A = _uniform(gen, batch * k * ld, dtype)
    cols = A.view(batch, k, ld)
    cols[:, :, :k] /= k
    d = torch.diagonal(cols[:, :, :k], dim1=1, dim2=2)
    d.mul_(0.5 * k).add_(1.5)
    return A


def _sizes(case):
    """Row and column counts of a variable-size batch: triangle orders log-uniform in [lo, hi],
    vector counts uniform in 1..nhi, drawn from the case's own number."""
    r = random.Random(case["sizes"])
    ks = [_log_int(r, case["lo"], case["hi"]) for _ in range(case["batch"])]
    vs = [r.randint(1, case["nhi"]) for _ in range(case["batch"])]
    return (ks, vs) if case["side"] == "L" else (vs, ks)


def _offsets(counts):
    out = [0]
    for c in counts:
        out.append(out[-1] + c)
    return out


def _inputs(case, seed):
    """The operands of a case as flat device tensors (A, B), B None for an inverse."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dtype, op = _dtype(case), case["op"]
    if op == "trtri":
        return _triangles(gen, case["n"], case["n"] + case["pad"], case["batch"], dtype), None
    if op == "trsm":
        m, n, batch, pad = case["m"], case["n"], case["batch"], case["pad"]
        k = m if case["side"] == "L" else n
        return (_triangles(gen, k, k + pad, batch, dtype),
                _uniform(gen, batch * n * (m + pad), dtype))
    ms, ns = _sizes(case)
    ks = ms if case["side"] == "L" else ns
    off = _offsets([k * k for k in ks])
    order = torch.tensor(ks, dtype=torch.int64, device="cuda")
    A = _uniform(gen, off[-1], dtype)
    A /= torch.repeat_interleave(order.to(dtype), order * order)
    start = torch.tensor(off[:-1], dtype=torch.int64, device="cuda")
    which = torch.repeat_interleave(torch.arange(len(ks), device="cuda"), order)
    row = torch.arange(int(which.numel()), device="cuda") - torch.tensor(
        _offsets(ks)[:-1], dtype=torch.int64, device="cuda")[which]
    at = start[which] + row * (order[which] + 1)
    A[at] = A[at] * (0.5 * order[which]).to(dtype) + 1.5
    return A, _uniform(gen, sum(m * n for m, n in zip(ms, ns)), dtype)


def _pointers(t, offsets):
    base, size = t.data_ptr(), t.element_size()
    return torch.tensor([base + size * o for o in offsets], dtype=torch.int64, device="cuda")


def prepare(case, seed):
    handle = rb.Handle()
    rb.check(handle.set_stream(torch.cuda.current_stream().cuda_stream))
    A, B = _inputs(case, seed)
    s = dict(case, handle=handle, A=A, B=B)
    if case["op"] == "vbatched":
        ms, ns = _sizes(case)
        ks = ms if case["side"] == "L" else ns
        i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
        s.update(ms=i32(ms), ns=i32(ns), lda=i32(ks), ldb=i32(ms),
                 pa=_pointers(A, _offsets([k * k for k in ks])[:-1]),
                 pb=_pointers(B, _offsets([m * n for m, n in zip(ms, ns)])[:-1]))
    elif case["op"] == "trtri":
        n, ld = case["n"], case["n"] + case["pad"]
        s["X"] = torch.zeros_like(A)
        s["out"] = s["X"].view(case["batch"], n, ld)[:, :, :n]
    else:
        m, n, pad, batch = case["m"], case["n"], case["pad"], case["batch"]
        k = m if case["side"] == "L" else n
        s["out"] = B.view(batch, n, m + pad)[:, :, :m]
        if case["form"] == "pointers":
            s["pa"] = _pointers(A, [b * k * (k + pad) for b in range(batch)])
            s["pb"] = _pointers(B, [b * n * (m + pad) for b in range(batch)])
    return s


def run(s):
    """One call; the solution (or the inverse) as [batch, column, row], a variable-size batch's as
    the flat buffer that holds its instances back to back."""
    h, prec, op = s["handle"], s["prec"], s["op"]
    if op == "vbatched":
        rb.check(rb.trsm_vbatched(h, s["side"], s["uplo"], s["trans"], s["diag"],
                                  s["ms"].data_ptr(), s["ns"].data_ptr(), 1.0, s["pa"].data_ptr(),
                                  s["lda"].data_ptr(), s["pb"].data_ptr(), s["ldb"].data_ptr(),
                                  s["batch"], precision=prec))
        return s["B"]
    if op == "trtri":
        n, ld = s["n"], s["n"] + s["pad"]
        if s["batch"] == 1:
            rb.check(rb.trtri(h, s["uplo"], s["diag"], n, s["A"].data_ptr(), ld,
                              s["X"].data_ptr(), ld, precision=prec))
        else:
            rb.check(rb.trtri_strided_batched(h, s["uplo"], s["diag"], n, s["A"].data_ptr(), ld,
                                              n * ld, s["X"].data_ptr(), ld, n * ld, s["batch"],
                                              precision=prec))
        return s["out"]
    m, n, batch = s["m"], s["n"], s["batch"]
    k = m if s["side"] == "L" else n
    lda, ldb = k + s["pad"], m + s["pad"]
    what = (h, s["side"], s["uplo"], s["trans"], s["diag"], m, n, s["alpha"])
    if s["form"] == "single":
        st = rb.trsm(*what, s["A"].data_ptr(), lda, s["B"].data_ptr(), ldb, precision=prec)
    elif s["form"] == "strided":
        st = rb.trsm_strided_batched(*what, s["A"].data_ptr(), lda, k * lda, s["B"].data_ptr(),
                                     ldb, n * ldb, batch, precision=prec)
    else:
        st = rb.trsm_batched(*what, s["pa"].data_ptr(), lda, s["pb"].data_ptr(), ldb, batch,
                             precision=prec)
    rb.check(st)
    return s["out"]


def work(case):
    """Triangle read once, right-hand sides read and written once; k^2 operations a vector (as the
    reference counts trsm), n^3 / 3 an inverse."""
    size = 8 if case["prec"] == "d" else 4
    if case["op"] == "trtri":
        n, b = case["n"], case["batch"]
        return {"bytes": size * b * (n * (n + 1) / 2 + n * n), "flops": b * n ** 3 / 3}
    if case["op"] == "vbatched":
        ms, ns = _sizes(case)
    else:
        ms, ns = [case["m"]], [case["n"]]
    scale = 1 if case["op"] == "vbatched" else case["batch"]
    ks = ms if case["side"] == "L" else ns
    return {"bytes": scale * size * sum(k * (k + 1) / 2 + 2 * m * n
                                        for k, m, n in zip(ks, ms, ns)),
            "flops": scale * sum(float(k) * m * n for k, m, n in zip(ks, ms, ns))}


def _solve(case, A, B, alpha):
    """op(A) X = alpha B or X op(A) = alpha B for mathematical matrices A [.., k, k], B [.., m, n]."""
    upper, left = case["uplo"] == "U", case["side"] == "L"
    if case["trans"] == "T":
        A, upper = A.transpose(-1, -2), not upper
    if A.dim() == 2 or A.shape[0] == 1:
        return torch.linalg.solve_triangular(A, alpha * B, upper=upper, left=left,
                                             unitriangular=case["diag"] == "U")
    # a batch: substitution on the vectors as rows, X [batch, vector, k], all instances at a time
    if not left:
        A, upper = A.transpose(1, 2), not upper
    X = (alpha * (B.transpose(1, 2) if left else B)).contiguous()
    k = A.shape[1]
    for i in (reversed(range(k)) if upper else range(k)):
        if case["diag"] == "N":
            X[:, :, i] /= A[:, i, i, None]
        rest = slice(0, i) if upper else slice(i + 1, k)
        X[:, :, rest] -= X[:, :, i, None] * A[:, rest, i][:, None, :]
    return X.transpose(1, 2) if left else X


def exact(case, seed):
    A, B = _inputs(case, seed)
    A = A.double()
    if case["op"] == "vbatched":
        B = B.double()
        ms, ns = _sizes(case)
        a = b = 0
        for m, n in zip(ms, ns):
            k = m if case["side"] == "L" else n
            x = _solve(case, A[a:a + k * k].view(k, k).T, B[b:b + m * n].view(n, m).T, 1.0)
            B[b:b + m * n] = x.T.reshape(-1)
            a, b = a + k * k, b + m * n
        return B
    if case["op"] == "trtri":
        n, batch = case["n"], case["batch"]
        M = A.view(batch, n, n + case["pad"])[:, :, :n].transpose(1, 2)
        eye = torch.eye(n, dtype=torch.float64, device="cuda").expand(batch, n, n)
        inv = _solve(dict(case, side="L", trans="N"), M, eye, 1.0)
        inv = torch.triu(inv) if case["uplo"] == "U" else torch.tril(inv)
        return inv.transpose(1, 2).contiguous()
    m, n, batch, pad = case["m"], case["n"], case["batch"], case["pad"]
    k = m if case["side"] == "L" else n
    M = A.view(batch, k, k + pad)[:, :, :k].transpose(1, 2)
    R = B.double().view(batch, n, m + pad)[:, :, :m].transpose(1, 2)
    return _solve(case, M, R, case["alpha"]).transpose(1, 2).contiguous()
