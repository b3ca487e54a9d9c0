"""Variable-size batched GEMM (dmk_gemm_vbatch_{d,z}, the dmrg_Xgemm_vbatch boundary) against
numpy on the same inputs."""
import numpy as np
import pytest

import dmrgpp_amd as dm


def _op(x, t):
    return {"N": x, "T": x.T, "C": x.conj().T}[t]


def _run(transa, transb, cplx, alpha, beta, seed):
    rng = np.random.default_rng(seed)
    dt = np.complex128 if cplx else np.float64
    # Mixed shapes: tiny, ragged, tile-crossing, k = 0 and an empty entry.
    shapes = [(1, 1, 1), (7, 5, 3), (64, 64, 64), (65, 130, 17), (200, 33, 129), (3, 90, 0),
              (0, 4, 5), (150, 1, 70)]
    groups, keep, want, dev = [], [], [], []
    for (m, n, k) in shapes:
        ra, ca = (k, m) if transa != "N" else (m, k)
        rb, cb = (n, k) if transb != "N" else (k, n)
        lda, ldb, ldc = ra + 3, rb + 1, m + 2

        def rnd(r, c, ld):
            x = rng.uniform(-1, 1, (ld, max(c, 1)))
            if cplx:
                x = x + 1j * rng.uniform(-1, 1, (ld, max(c, 1)))
            return np.asfortranarray(x.astype(dt))
        entries = []
        for _ in range(2):
            A, B, C = rnd(ra, ca, max(lda, 1)), rnd(rb, cb, max(ldb, 1)), rnd(m, n, max(ldc, 1))
            if beta == 0:
                C[:] = np.nan  # must not be read
            Av, Bv = A[:ra, :ca], B[:rb, :cb]
            Cw = C.copy()
            if m and n:
                prod = _op(Av, transa) @ _op(Bv, transb) if k else np.zeros((m, n), dt)
                Cw[:m, :n] = alpha * prod + (beta * C[:m, :n] if beta != 0 else 0)
            dA = dm.DeviceArray.from_host(A.ravel(order="F").view(np.float64))
            dB = dm.DeviceArray.from_host(B.ravel(order="F").view(np.float64))
            dC = dm.DeviceArray.from_host(C.ravel(order="F").view(np.float64))
            dev += [dA, dB, dC]
            want.append((dC, Cw, m, n))
            entries.append((dA.ptr, dB.ptr, dC.ptr))
        groups.append((m, n, k, max(lda, 1), max(ldb, 1), max(ldc, 1), entries))
    dm.gemm_vbatch(transa, transb, groups, alpha=alpha, beta=beta, cplx=cplx)
    for dC, Cw, m, n in want:
        got = dC.download().view(dt).reshape(Cw.shape, order="F")
        if m and n:
            ref = Cw[:m, :n]
            err = np.abs(got[:m, :n] - ref).max() / max(1.0, np.abs(ref).max())
            assert err < 1e-13, (m, n, err)


def test_vbatch_rejects_bad_arguments():
    one = (dm.ctypes.c_int * 1)(4)
    ptr = (dm.ctypes.c_void_p * 1)(0)
    L = dm.lib()
    a = dm.ctypes.addressof
    assert L.dmk_gemm_vbatch_d(b"X", b"N", a(one), a(one), a(one), 1.0, a(ptr), a(one), a(ptr),
                               a(one), 0.0, a(ptr), a(one), 1, a(one)) == -1
    assert b"transa" in L.dmk_last_error()
    small = (dm.ctypes.c_int * 1)(2)
    assert L.dmk_gemm_vbatch_d(b"N", b"N", a(one), a(one), a(one), 1.0, a(ptr), a(small),
                               a(ptr), a(one), 0.0, a(ptr), a(one), 1, a(one)) == -1
    assert b"leading dimension" in L.dmk_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("transa,transb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-0.5, 1.0), (2.0, 0.25)])
def test_gpu_vbatch_real(transa, transb, alpha, beta):
    _run(transa, transb, False, alpha, beta, seed=ord(transa) * 7 + ord(transb) + int(10 * alpha))


@pytest.mark.gpu
@pytest.mark.parametrize("transa,transb", [("N", "N"), ("C", "N"), ("T", "C")])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (0.5 - 1j, 0.3 + 0.2j)])
def test_gpu_vbatch_complex(transa, transb, alpha, beta):
    _run(transa, transb, True, alpha, beta, seed=7)


@pytest.mark.gpu
def test_gpu_vbatch_alpha_zero_scales_c_only():
    # alpha = 0: C = beta C, A and B (NaN here) are not used.
    m = n = k = 20
    A = np.full((m, k), np.nan)
    C = np.arange(m * n, dtype=float).reshape(m, n, order="F")
    dA = dm.DeviceArray.from_host(A.ravel(order="F"))
    dC = dm.DeviceArray.from_host(C.ravel(order="F"))
    dm.gemm_vbatch("N", "N", [(m, n, k, m, k, m, [(dA.ptr, dA.ptr, dC.ptr)])], alpha=0.0,
                   beta=3.0)
    np.testing.assert_array_equal(dC.download().reshape(m, n, order="F"), 3.0 * C)


@pytest.mark.gpu
@pytest.mark.parametrize("cplx", [False, True])
def test_gpu_vbatch_alpha_zero_takes_any_contraction(cplx):
    # With alpha = 0 the operands are not read, whatever k says; a product that long is refused by
    # the entry point's limit, and C is left alone.
    w = 2 if cplx else 1
    m, n, k = 3, 2, (1 << 21) + 1
    C = np.random.default_rng(6).uniform(-1, 1, w * m * n)
    dA, dC = dm.DeviceArray(1), dm.DeviceArray.from_host(C)
    group = [(m, n, k, m, k, m, [(dA.ptr, dA.ptr, dC.ptr)])]
    with pytest.raises(dm.DmkError, match="contraction is longer than 2097152"):
        dm.gemm_vbatch("N", "N", group, alpha=1.0, beta=3.0, cplx=cplx)
    np.testing.assert_array_equal(dC.download(), C)
    dm.gemm_vbatch("N", "N", group, alpha=0.0, beta=3.0, cplx=cplx)
    np.testing.assert_array_equal(dC.download(), 3.0 * C)


@pytest.mark.gpu
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("transa,transb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
def test_gpu_vbatch_large_batch_tiles(transa, transb, cplx):
    # Enough tiles for the 64 x 64 kernel (2112 of them), k with and without a remainder of a 16-element
    # chunk and past the four chunks in flight, an odd base address.
    rng = np.random.default_rng(3)
    w = 2 if cplx else 1
    dt = np.complex128 if cplx else np.float64
    tall = 64 * 64
    shapes = [(tall, 64 * 33, 17), (129, 63, 15), (33, 65, 16), (64, 64, 47), (31, 97, 64), (1, 1, 100)]
    buf = rng.uniform(-1, 1, w * (tall * 128 + 1))
    dX = dm.DeviceArray.from_host(buf)
    view = buf[1:1 + w * tall * 128].view(dt)
    groups, outs = [], []
    for m, n, k in shapes:
        lda, ldb = (k if transa != "N" else m) + 1, (n if transb != "N" else k) + 2
        A = view[:lda * (m if transa != "N" else k)].reshape((lda, -1), order="F")[:lda - 1]
        B = view[:ldb * (k if transb != "N" else n)].reshape((ldb, -1), order="F")[:ldb - 2]
        dC = dm.DeviceArray(w * m * n)
        groups.append((m, n, k, lda, ldb, m, [(dX.ptr + 8, dX.ptr + 8, dC.ptr)]))
        outs.append((dC, _op(A, transa) @ _op(B, transb)))
    dm.gemm_vbatch(transa, transb, groups, cplx=cplx)
    for (dC, want), (m, n, k) in zip(outs, shapes):
        got = dC.download().view(dt).reshape((m, n), order="F")
        # k products of at most 1 (2 for complex), k + 2 roundings each way.
        assert np.abs(got - want).max() <= 2 * w * w * k * (k + 2) * 2.0 ** -53


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 8, 9, 512, 513, 4097, 40000])
def test_gpu_vbatch_many_small_entries(count):
    # One run per entry: lists of 1 to 5000 runs per XCD (one, two and three steps of the search), sizes
    # of one tile and, every 97th entry, several.
    rng = np.random.default_rng(count)
    i = np.arange(count)
    m, n, k = 1 + i % 5, 1 + i % 3, i % 4
    m[::97] += 60
    A = rng.uniform(-1, 1, int((m * np.maximum(k, 1)).sum()))
    B = rng.uniform(-1, 1, int((n * np.maximum(k, 1)).sum()))
    dA, dB, dC = dm.DeviceArray.from_host(A), dm.DeviceArray.from_host(B), dm.DeviceArray(int((m * n).sum()))
    dC.upload(np.full(dC.size, np.nan))
    oa, ob, oc = (np.concatenate([[0], np.cumsum(v)]) for v in
                  (m * np.maximum(k, 1), n * np.maximum(k, 1), m * n))
    dm.gemm_vbatch("N", "T", [(int(m[e]), int(n[e]), int(k[e]), int(m[e]), int(n[e]), int(m[e]),
                               [(dA.ptr + 8 * int(oa[e]), dB.ptr + 8 * int(ob[e]), dC.ptr + 8 * int(oc[e]))])
                              for e in range(count)])
    got = dC.download()
    for e in range(count):
        a = A[oa[e]:oa[e + 1]].reshape((-1, m[e]))[:k[e]]
        b = B[ob[e]:ob[e + 1]].reshape((-1, n[e]))[:k[e]]
        # At most three products of at most 1.
        assert np.abs(got[oc[e]:oc[e + 1]].reshape((n[e], m[e])) - b.T @ a).max() <= 24 * 2.0 ** -53


@pytest.mark.gpu
@pytest.mark.parametrize("wide", [False, True])
def test_gpu_vbatch_output_over_input_and_wide_rows(wide):
    # C in the memory of A (computed through a workspace), and a leading dimension past 2^21.
    rng = np.random.default_rng(4)
    m, n, k = 5, 3, 4
    ld = (1 << 21) + 3 if wide else m
    X = rng.uniform(-1, 1, ld * 4)
    B = rng.uniform(-1, 1, (k, n))
    dX, dB = dm.DeviceArray.from_host(X), dm.DeviceArray.from_host(B.ravel(order="F"))
    A = X.reshape((ld, 4), order="F")[:m, :k].copy()
    dm.gemm_vbatch("N", "N", [(m, n, k, ld, k, ld, [(dX.ptr, dB.ptr, dX.ptr)])], alpha=2.0, beta=0.5)
    got = dX.download().reshape((ld, 4), order="F")
    want = 2.0 * A @ B + 0.5 * A[:, :n]
    assert np.abs(got[:m, :n] - want).max() <= 16 * (k + 3) * 2.0 ** -53
    np.testing.assert_array_equal(got[:m, n:], A[:, n:])
    if wide:
        np.testing.assert_array_equal(got[m:], X.reshape((ld, 4), order="F")[m:])


@pytest.fixture(scope="module")
def wide_buffers():
    """Device memory for two matrices of 70 complex columns 2^21 + 3 apart."""
    a, b = (dm.DeviceArray(2 * 70 * ((1 << 21) + 3)) for _ in range(2))
    yield a, b
    a.free()
    b.free()


@pytest.mark.gpu
@pytest.mark.parametrize("transa,transb,cplx", [(a, b, c) for c in (False, True) for a in "NTC" for b in "NTC"
                                                if c or "C" not in (a, b)])
@pytest.mark.parametrize("count", [1, 1100])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("k", [4, 16, 70])
def test_gpu_vbatch_tiles_and_offsets(wide_buffers, k, wide, count, transa, transb, cplx):
    # 32- and 64-wide tiles (1 and 1100 tiles of 64 x 64) with 32- and 64-bit operand offsets (leading
    # dimensions past 2^21), every transpose, alpha and beta, and contractions of a remainder
    # alone, one whole chunk, and more chunks than are in flight with a remainder.
    rng = np.random.default_rng(k)
    w, dt = (2, np.complex128) if cplx else (1, np.float64)
    alpha, beta = (0.5 - 0.25j, 2.0 + 1.0j) if cplx else (-0.5, 2.0)
    m, n = 61, 63
    stored = []
    for dev, t, shape in zip(wide_buffers, (transa, transb), ((m, k), (k, n))):
        r, c = shape if t == "N" else shape[::-1]
        ld = (1 << 21) + 3 if wide else r + 1
        x = rng.uniform(-1, 1, (c, r * w))  # by columns
        for j in range(c):
            dm._check(dm.lib().dmk_memcpy_h2d(dev.ptr + 8 * w * ld * j, x[j].ctypes.data, x[j].nbytes), "copy")
        stored.append((dev.ptr, ld, _op(x.view(dt).T, t)))
    (pa, lda, A), (pb, ldb, B) = stored
    C = rng.uniform(-1, 1, (count, n, m * w))
    dC = dm.DeviceArray.from_host(C.ravel())
    dm.gemm_vbatch(transa, transb, [(m, n, k, lda, ldb, m, [(pa, pb, dC.ptr + e * C[0].nbytes)
                                                            for e in range(count)])],
                   alpha=alpha, beta=beta, cplx=cplx)
    got = dC.download().view(dt).reshape(count, n, m)
    want = alpha * (A @ B).T + beta * C.view(dt)
    # k products of parts at most 1 (w of them to a part of the result), w k + 4 roundings each way,
    # |alpha| < 1, and beta C at most 3 with four roundings.
    assert np.abs(got - want).max() <= 2 * w * (w * k * (w * k + 4) + 16) * 2.0 ** -53
