"""Kernel variants at the sizes where they can go wrong (edges of tiles, remainders, the smallest
and largest of their range), against the CPU oracle or a plain FP64 reference."""
import ctypes

import numpy as np
import pytest

import oracle as orc
import utopia_amd as ua

pytestmark = pytest.mark.gpu


def P(d):
    return ctypes.c_void_p(d.ptr)


def _rows_of_lengths(lengths, ncols, seed):
    rng = np.random.default_rng(seed)
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(ncols, k, replace=False)) for k in lengths]).astype(np.int32)
    return ua.Csr(rp, col, rng.standard_normal(col.size), (len(lengths), ncols))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("block_nnz", [1024, 2048])
def test_row_block_sums_in_column_order_at_every_length_and_alignment(ctx, dtype, block_nnz):
    # every length up to five 16-entry steps (one row after the other, so each LDS alignment
    # occurs), and the longest rows that one lane sums alone
    lengths = list(range(0, 83)) + [block_nnz + block_nnz // 4 - k for k in range(4)] + [1, 0, 35]
    A = _rows_of_lengths(lengths, 6000, 5)
    x = ua.gen_uniform(6, A.shape[1]).astype(dtype)
    D = ua.DeviceCsr(ctx, A, dtype, block_nnz)
    xd, yd = ua.DeviceArray.from_numpy(ctx, x), ua.DeviceArray(ctx, A.shape[0], dtype)
    D.spmv(xd, yd)
    ref = orc.spmv(A, x) if dtype == np.float64 else orc.spmv_f32(A, x)
    assert np.array_equal(yd.numpy(), ref)


def _csr_of(ctx, m):
    C = ua.csr_from_raw(ctx, m)
    ua.check(ua.lib().uhip_csr_free(ctx.h, ctypes.byref(m)))
    return C


def _product_equals_oracle(ctx, A, B):
    DA, DB, C = ua.DeviceCsr(ctx, A), ua.DeviceCsr(ctx, B), ua.uhip_csr()
    ua.check(ua.lib().uhip_csr_spgemm(ctx.h, DA.ref, DB.ref, ctypes.byref(C)))
    Ch = _csr_of(ctx, C)
    rp, col, val, shape = orc.spgemm(A, B)
    assert Ch.shape == shape and np.array_equal(Ch.rowptr, rp)
    assert np.array_equal(Ch.col, col) and np.array_equal(Ch.val, val)


@pytest.mark.parametrize("b_rows", [3, 8, 9, 16, 17, 40])
def test_spgemm_rows_around_the_hash_tables_limits(ctx, b_rows):
    # rows of C with few columns, with 55 .. 58 and 447 .. 450 (7/8 of the 64- and the 512-slot table, more than
    # either is filled to), with more, and empty ones; the mean length of B's rows picks the lanes a row of C has
    rng = np.random.default_rng(b_rows)
    nb, m = 700, 900
    B = _rows_of_lengths([b_rows] * (nb - 2) + [0, 1], m, 31)
    per_k = [np.zeros(0, np.int32)]
    union = set()
    order = rng.permutation(nb)
    want = [1, 2, 20, 55, 56, 57, 58, 447, 448, 449, 450]
    for target in want:  # add rows of B until the target is reached: neighbours of it occur too
        union, ks = set(), []
        for k in order:
            new = union | set(B.col[B.rowptr[k]:B.rowptr[k + 1]].tolist())
            if len(new) > target + 2:
                continue
            union = new
            ks.append(k)
            if len(ks) * b_rows > 7000 or len(union) >= target:
                break
        per_k.append(np.sort(np.array(ks, np.int32)))
    per_k += [np.arange(0, nb, 5, dtype=np.int32)] * 3 + [np.zeros(0, np.int32)]
    per_k += [np.sort(rng.choice(nb, 7, replace=False)).astype(np.int32) for _ in range(200)]
    rp = np.concatenate([[0], np.cumsum([k.size for k in per_k])]).astype(np.int32)
    col = np.concatenate(per_k).astype(np.int32)
    A = ua.Csr(rp, col, rng.standard_normal(col.size), (len(per_k), nb))
    _product_equals_oracle(ctx, A, B)


@pytest.mark.parametrize("b_rows", [5, 12, 30])
@pytest.mark.parametrize("kind", ["few duplicates", "many duplicates"])
def test_spgemm_rows_around_the_limits_of_the_tables_and_classes(ctx, b_rows, kind):
    # rows of C with 38 .. 42 and 254 .. 258 columns (the 64- and the 512-slot table are filled to 40 and 256), by few
    # candidates a column (rows of B that do not meet: the next place is the sorting) and by many (every row of B twice,
    # shifted by one: the larger table), and rows whose candidates lie around the sorting's classes at 256 and 1024
    rng = np.random.default_rng(b_rows)
    nb, m = 1200, 40000
    base = np.arange(nb) * b_rows % (m - b_rows - 1) if kind == "few duplicates" else np.arange(nb) // 2 + np.arange(nb) % 2
    lens = np.where(np.arange(nb) % 3 == 0, 1, b_rows)
    B = ua.Csr(np.r_[0, np.cumsum(lens)].astype(np.int32),
               np.concatenate([b + np.arange(k) for b, k in zip(base, lens)]).astype(np.int32),
               rng.standard_normal(lens.sum()), (nb, m))
    rows = []
    for target in [1, 3, 38, 39, 40, 41, 42, 120, 253, 254, 255, 256, 257, 258, 300]:
        cols, ks = set(), []
        for k in range(rng.integers(0, 50), nb):
            new = cols | set(range(base[k], base[k] + lens[k]))
            if len(new) > target:
                continue
            ks.append(k)
            cols = new
            if sum(lens[ks]) > 7900:
                break
        rows.append(ks)
    for cand in (255, 256, 257, 1023, 1024, 1025, 4095, 4096, 4097, 8000):
        ks, c = [], 0
        for k in range(nb):
            if c + lens[k] <= cand:
                ks.append(k)
                c += lens[k]
        rows.append(ks)
    rows += [[], [nb - 1]]
    col = np.concatenate([np.array(k, np.int32) for k in rows]).astype(np.int32)
    A = ua.Csr(np.r_[0, np.cumsum([len(k) for k in rows])].astype(np.int32), col, rng.standard_normal(col.size), (len(rows), nb))
    _product_equals_oracle(ctx, A, B)
    # the same rows among 2,000 short ones: the sample finds no reason to sort them all
    short = [[int(k)] for k in rng.integers(0, nb, 2000)]
    col = np.concatenate([np.array(k, np.int32) for k in rows + short]).astype(np.int32)
    A = ua.Csr(np.r_[0, np.cumsum([len(k) for k in rows + short])].astype(np.int32), col, rng.standard_normal(col.size),
               (len(rows) + 2000, nb))
    _product_equals_oracle(ctx, A, B)


@pytest.mark.parametrize("n", [1, 127, 129, 3000])
@pytest.mark.parametrize("band", [False, True])
def test_spgemm_of_long_rows_with_few_and_many_duplicates(ctx, n, band):
    # more than 1024 candidates in the longest row: sampled, and every row sorted (random columns), or not (a band)
    rng = np.random.default_rng(n)
    if band:
        B = _rows_of_lengths([1] * 60, 90, 2)
        B = ua.Csr(np.arange(0, 60 * 40 + 1, 40, dtype=np.int32),
                   (np.arange(60)[:, None] // 3 + np.arange(40)[None, :]).ravel().astype(np.int32),
                   rng.standard_normal(2400), (60, 90))
        A = _rows_of_lengths(rng.integers(28, 40, n).tolist(), 60, n)
    else:
        B = _rows_of_lengths(rng.integers(10, 60, 500).tolist(), 20000, 3)
        A = _rows_of_lengths(rng.integers(1, 40, n - 1).tolist() + [45], 500, n)
    _product_equals_oracle(ctx, A, B)


def test_spgemm_of_rows_with_unsorted_and_repeated_columns(ctx):
    rng = np.random.default_rng(4)
    B = _rows_of_lengths([6] * 60, 40, 32)
    B.col = rng.integers(0, 40, B.col.size).astype(np.int32)
    _product_equals_oracle(ctx, _rows_of_lengths([5] * 50, 60, 33), B)


@pytest.mark.parametrize("longest", [31, 32, 33, 511, 512, 513, 2000])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_transpose_of_columns_around_the_ordering_limits(ctx, longest, dtype):
    # a column of `longest` entries among short ones, columns of the lower halves, empty columns
    rng = np.random.default_rng(longest)
    n, m = 2100, 50
    cols = [np.sort(rng.choice(np.arange(10, 45), rng.integers(0, 3), replace=False)) for _ in range(n)]
    rows = np.sort(rng.choice(n, longest, replace=False))
    for r in rows:
        cols[r] = np.concatenate([[7], cols[r]])
    for r in rows[:longest // 2]:
        cols[r] = np.concatenate([[3], cols[r]])
    rp = np.concatenate([[0], np.cumsum([c.size for c in cols])]).astype(np.int32)
    col = np.concatenate(cols).astype(np.int32)
    # values that FP32 holds, so that one oracle serves both precisions
    A = ua.Csr(rp, col, rng.standard_normal(col.size).astype(np.float32).astype(np.float64), (n, m))
    D, T = ua.DeviceCsr(ctx, A, dtype), ua.uhip_csr()
    ua.check(ua.lib().uhip_csr_transpose(ctx.h, D.ref, ctypes.byref(T)))
    rp, col, val, shape = orc.transpose(A)
    vd = ua.DeviceArray(ctx, A.nnz, dtype)
    ua.check(ua.lib().uhip_memcpy_dtod(ctx.h, P(vd), ctypes.c_void_p(T.val), vd.n * vd.dtype.itemsize))
    v = vd.numpy()
    trp = np.zeros(m + 1, np.int32)
    tcol = np.zeros(A.nnz, np.int32)
    ua.check(ua.lib().uhip_memcpy_dtoh(ctx.h, ctypes.c_void_p(trp.ctypes.data), ctypes.c_void_p(T.rowptr), trp.nbytes))
    ua.check(ua.lib().uhip_memcpy_dtoh(ctx.h, ctypes.c_void_p(tcol.ctypes.data), ctypes.c_void_p(T.col), tcol.nbytes))
    assert (T.nrows, T.ncols) == shape and np.array_equal(trp, rp) and np.array_equal(tcol, col)
    assert np.array_equal(v, val.astype(dtype))
    ua.check(ua.lib().uhip_csr_free(ctx.h, ctypes.byref(T)))


@pytest.mark.parametrize("n", [2, 15, 16, 17, 64, 65, 127, 128, 129, 192, 257, 449, 1025])
def test_dense_factor_and_inverse_at_block_edges(ctx, n):
    # the 16- and 64-column blocks of the factor and the doubling steps of the inverse, with the last
    # block full, of one row, and missing; a leading dimension larger than n
    rng = np.random.default_rng(n)
    lda = n + 3
    M = rng.standard_normal((n, n))
    A = M @ M.T + n * np.eye(n)
    wide = np.zeros((n, lda))
    wide[:, :n] = A
    L = ua.lib()
    Ad, Inv = ua.DeviceArray.from_numpy(ctx, wide.ravel()), ua.DeviceArray(ctx, n * n)
    info = ctypes.c_int(-1)
    ua.check(L.uhip_dense_cholesky(ctx.h, n, P(Ad), lda, ctypes.byref(info)))
    assert info.value == 0
    got = Ad.numpy().reshape(n, lda)
    assert np.all(got[:, n:] == 0)
    ref = np.linalg.cholesky(A)
    # backward error of a factorisation: n eps |A| (Higham, Accuracy and Stability, thm 10.3)
    Lg = np.tril(got[:, :n])
    assert np.abs(Lg @ Lg.T - A).max() <= 2 * n * 2.3e-16 * np.abs(A).max()
    assert np.abs(Lg - ref).max() <= 1e-12 * np.abs(ref).max()
    ua.check(L.uhip_dense_cholesky_inverse(ctx.h, n, P(Ad), lda, P(Inv)))
    Ainv = Inv.numpy().reshape(n, n)
    assert np.array_equal(Ainv, Ainv.T)
    assert np.abs(Ainv @ A - np.eye(n)).max() <= 1e-12


@pytest.mark.parametrize("n", [1, 64, 65, 128, 129, 200, 449, 1025])
def test_dense_inverse_in_the_factors_own_memory(ctx, n):
    # Ainv is L's buffer: the same bits as from two buffers, at sizes with none to five doubling steps
    # and several column tiles a step
    rng = np.random.default_rng(n)
    M = rng.standard_normal((n, n))
    A = M @ M.T + n * np.eye(n)
    L = ua.lib()
    Ad, Inv, info = ua.DeviceArray.from_numpy(ctx, A.ravel()), ua.DeviceArray(ctx, n * n), ctypes.c_int(-1)
    ua.check(L.uhip_dense_cholesky(ctx.h, n, P(Ad), n, ctypes.byref(info)))
    assert info.value == 0
    ua.check(L.uhip_dense_cholesky_inverse(ctx.h, n, P(Ad), n, P(Inv)))
    ua.check(L.uhip_dense_cholesky_inverse(ctx.h, n, P(Ad), n, P(Ad)))
    assert np.array_equal(Ad.numpy(), Inv.numpy())
    assert np.abs(Inv.numpy().reshape(n, n) @ A - np.eye(n)).max() <= 1e-12


@pytest.mark.parametrize("n", [64, 130, 200])
@pytest.mark.parametrize("kind", ["scaled", "illconditioned"])
def test_dense_factor_and_inverse_of_badly_scaled_and_conditioned_matrices(ctx, n, kind):
    # rows scaled over 120 decades (Cholesky's rounding does not depend on a diagonal scaling), and a condition of
    # 1e10. In the scaling that makes the diagonal 1: |L L^T - A| <= (n + 1) eps (Higham, thm 10.3), and the
    # inverse's error within n times cond(A) times that
    rng = np.random.default_rng(n)
    if kind == "scaled":
        M = rng.standard_normal((n, n))
        d = 10.0 ** rng.uniform(-60, 60, n)
        A = (M @ M.T + n * np.eye(n)) * d[:, None] * d[None, :]
    else:
        Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
        A = (Q * np.logspace(0, -10, n)) @ Q.T
        A = (A + A.T) / 2
    L = ua.lib()
    Ad, Inv, info = ua.DeviceArray.from_numpy(ctx, A.ravel()), ua.DeviceArray(ctx, n * n), ctypes.c_int(-1)
    ua.check(L.uhip_dense_cholesky(ctx.h, n, P(Ad), n, ctypes.byref(info)))
    assert info.value == 0
    ua.check(L.uhip_dense_cholesky_inverse(ctx.h, n, P(Ad), n, P(Inv)))
    s = np.sqrt(np.diag(A))
    F = np.tril(Ad.numpy().reshape(n, n)) / s[:, None]
    C = A / s[:, None] / s[None, :]
    eps = 2.3e-16
    assert np.abs(F @ F.T - C).max() <= 2 * (n + 1) * eps
    X = Inv.numpy().reshape(n, n) * s[:, None] * s[None, :]
    assert np.linalg.norm(X @ C - np.eye(n), 2) <= 2 * n * n * eps * np.linalg.cond(C)


@pytest.mark.parametrize("n,held", [(3, [1]), (64, [0, 17]), (130, [5, 63, 64, 128]), (200, [70, 199])])
def test_dense_factor_with_infinite_diagonal_entries(ctx, n, held):
    # such a row is held at zero: its column of the factor is zero below an infinite pivot, and the inverse is that of
    # the other rows
    rng = np.random.default_rng(n)
    M = rng.standard_normal((n, n))
    A = M @ M.T + n * np.eye(n)
    A[held, held] = np.inf
    L = ua.lib()
    Ad, Inv, info = ua.DeviceArray.from_numpy(ctx, A.ravel()), ua.DeviceArray(ctx, n * n), ctypes.c_int(-1)
    ua.check(L.uhip_dense_cholesky(ctx.h, n, P(Ad), n, ctypes.byref(info)))
    assert info.value == 0
    F = np.tril(Ad.numpy().reshape(n, n))
    free = np.setdiff1d(np.arange(n), held)
    B = A[np.ix_(free, free)]
    assert np.all(np.isinf(np.diag(F)[held])) and all(np.all(F[k + 1:, k] == 0) for k in held)
    assert np.abs(F[np.ix_(free, free)] - np.linalg.cholesky(B)).max() <= 1e-12 * np.sqrt(B.max())
    ua.check(L.uhip_dense_cholesky_inverse(ctx.h, n, P(Ad), n, P(Inv)))
    X = Inv.numpy().reshape(n, n)
    assert np.all(X[held] == 0) and np.all(X[:, held] == 0)
    assert np.abs(X[np.ix_(free, free)] @ B - np.eye(free.size)).max() <= 1e-12


@pytest.mark.parametrize("bad", [0, 15, 16, 40, 63, 64, 100, 129])
def test_dense_factor_reports_the_first_bad_pivot(ctx, bad):
    n = 130
    A = np.eye(n) * 4
    A[bad, bad] = -1.0
    A[n - 1, n - 1] = -2.0
    Ad, info = ua.DeviceArray.from_numpy(ctx, A.ravel()), ctypes.c_int()
    ua.check(ua.lib().uhip_dense_cholesky(ctx.h, n, P(Ad), n, ctypes.byref(info)))
    assert info.value == bad + 1


def _jacobi_cg(A, b, atol, max_steps):
    """The loop in FP64 numpy: (x, iterations, |r|, reason)."""
    S, d = A.to_scipy(), 1.0 / A.to_scipy().diagonal()
    x, r = np.zeros_like(b), b.copy()
    p = d * r
    rz, norm = r @ p, np.inf
    for j in range(max_steps):
        Ap = S @ p
        with np.errstate(divide="ignore", invalid="ignore"):
            alpha = rz / (p @ Ap)
        if not np.isfinite(alpha):
            return x, j, norm, 2
        x = x + alpha * p
        r = r - alpha * Ap
        norm = np.sqrt(r @ r)
        if norm <= atol:
            return x, j + 1, norm, 1
        z = d * r
        rz_new = r @ z
        p = z + rz_new / rz * p
        rz = rz_new
    return x, max_steps, norm, 0


@pytest.mark.parametrize("dims,fmt", [((1, 1), None), ((3, 2), None), ((17, 15), ua.FMT_ROWBLOCK), ((64, 64), ua.FMT_SELL64),
                                      ((255, 257), None), ((1100, 1000), None)])
@pytest.mark.parametrize("max_steps", [1, 3, 40])
def test_jacobi_cg_iterations_on_the_device(ctx, dims, fmt, max_steps):
    # one row, fewer rows than a wavefront, several rows a thread (1.1M), partial sums added by the
    # consumer and, over 2048 workgroups, by the finishing kernel
    A = ua.gen_stencil(ua.STENCIL_2D5, *dims)
    n = A.shape[0]
    b = ua.gen_uniform(9, n)
    ref, its, norm, why = _jacobi_cg(A, b, 1e-13, max_steps)
    D = ua.DeviceCsr(ctx, A, fmt=fmt)
    d = 1.0 / A.to_scipy().diagonal()
    xd, rd, pd, Apd, dd = (ua.DeviceArray.from_numpy(ctx, v) for v in (np.zeros(n), b, d * b, np.zeros(n), d))
    rz = ua.DeviceArray.from_numpy(ctx, np.array([b @ (d * b)]))
    steps, rn, reason = ctypes.c_int64(), ctypes.c_double(), ctypes.c_int()
    ua.check(ua.lib().uhip_cg_jacobi_f64(ctx.h, D.ref, P(dd), P(xd), P(rd), P(pd), P(Apd), P(rz), 1e-13, max_steps,
                                         ctypes.byref(steps), ctypes.byref(rn), ctypes.byref(reason)))
    assert (steps.value, reason.value) == (its, why)
    # rounding grows with the iterations done (at most 40): 1e3 eps a step
    assert np.linalg.norm(xd.numpy() - ref) <= 40 * 1e3 * 2.3e-16 * np.linalg.norm(ref)
    if why != 1:
        assert abs(rn.value - norm) <= 40 * 1e3 * 2.3e-16 * np.linalg.norm(b)
    else:
        assert rn.value <= 1e-13


@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("offsets", [(0,), (1, 3), (1, 2, 7, 9, 30), tuple(range(1, 14)), tuple(range(1, 15)) + (200,)])
@pytest.mark.parametrize("n", [1, 255, 256, 257, 5000])
def test_jacobi_cg_on_a_diagonal_plan(ctx, n, offsets, symmetric):
    # the update in the next product: 1 to 31 diagonals (8- to 32-bit masks, more than one round of loads), both
    # layouts; x, r and p as the iterations leave them, after odd and even counts. The matrix is near the identity, so
    # an iteration's values hold to a few hundred eps; p after several steps is small: against |b|.
    import scipy.sparse as sp
    rng = np.random.default_rng(n)
    S = sp.diags([rng.uniform(1, 2, n)], [0])
    for o in offsets:
        if 0 < o < n:
            lo = rng.uniform(-0.02, 0.02, n - o)
            S = S + sp.diags([lo, lo if symmetric else rng.uniform(-0.02, 0.02, n - o)], [-o, o])
    A = ua.Csr.from_scipy(S.tocsr())
    S, d, b = S.tocsr(), 1.0 / S.diagonal(), rng.uniform(-1, 1, n)
    D = ua.DeviceCsr(ctx, A, fmt=ua.FMT_DIA)
    for steps in (1, 2, 3, 8):
        x, r, p = np.zeros(n), b.copy(), d * b
        rz = r @ p
        done = 0
        while done < steps:
            Ap = S @ p
            alpha = rz / (p @ Ap)
            x, r = x + alpha * p, r - alpha * Ap
            rz, old = r @ (d * r), rz
            p = d * r + rz / old * p
            done += 1
            if np.sqrt(r @ r) <= 1e-4:
                break
        xd, rd, pd, Apd, dd, rzd = (ua.DeviceArray.from_numpy(ctx, v)
                                    for v in (np.zeros(n), b, d * b, np.zeros(n), d, np.array([b @ (d * b)])))
        its, rn, reason = ctypes.c_int64(), ctypes.c_double(), ctypes.c_int()
        ua.check(ua.lib().uhip_cg_jacobi_f64(ctx.h, D.ref, P(dd), P(xd), P(rd), P(pd), P(Apd), P(rzd), 1e-4, steps,
                                             ctypes.byref(its), ctypes.byref(rn), ctypes.byref(reason)))
        assert its.value == done
        for got, ref in ((xd, x), (rd, r), (pd, p)):
            assert np.linalg.norm(got.numpy() - ref) <= 8 * 1e3 * 2.3e-16 * np.linalg.norm(b)


def test_jacobi_cg_stops_on_a_step_that_is_not_finite(ctx):
    # p.Ap = 0 (a zero operator): alpha is infinite, nothing moves; and through the solver the status
    # that the host-paced loop gave
    n = 300
    A = ua.Csr(np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.zeros(n), (n, n))
    b = ua.gen_uniform(3, n)
    D = ua.DeviceCsr(ctx, A)
    xd, rd, pd, Apd, dd = (ua.DeviceArray.from_numpy(ctx, v) for v in (np.ones(n), b, b, np.zeros(n), np.ones(n)))
    rz = ua.DeviceArray.from_numpy(ctx, np.array([b @ b]))
    steps, rn, reason = ctypes.c_int64(), ctypes.c_double(), ctypes.c_int()
    ua.check(ua.lib().uhip_cg_jacobi_f64(ctx.h, D.ref, P(dd), P(xd), P(rd), P(pd), P(Apd), P(rz), 1e-9, 50,
                                         ctypes.byref(steps), ctypes.byref(rn), ctypes.byref(reason)))
    assert (steps.value, reason.value) == (0, 2)
    assert np.array_equal(xd.numpy(), np.ones(n)) and np.array_equal(rd.numpy(), b)


@pytest.mark.parametrize("max_it", [0, 5, 500])
def test_jacobi_cg_status_with_and_without_printing(ctx, max_it, capfd):
    A = ua.gen_stencil(ua.STENCIL_2D5, 30, 20)
    b = ua.gen_uniform(5, A.shape[0])
    got = []
    for verbose in (0, 1):
        s = ua.ConjugateGradient(ctx, "jacobi", atol=1e-8, rtol=1e-30, stol=1e-30, max_it=max_it, verbose=verbose)
        x = s.solve(A, b)
        got.append((x, s.status))
    (x0, s0), (x1, s1) = got
    assert s0["iterates"] == s1["iterates"] and s0["reason"] == s1["reason"]
    assert s0["iterates"] == (max_it if max_it < 500 else s0["iterates"]) and s0["reason"] == (-5 if max_it < 500 else 2)
    assert np.linalg.norm(x0 - x1) <= 1e-12 * np.linalg.norm(x0)


def _obstacle(nx, ny, seed):
    A = ua.gen_stencil(ua.STENCIL_2D9, nx, ny, shift=1e-3)
    n = A.shape[0]
    return A, ua.gen_uniform(seed, n), -0.05 - 0.15 * ua.gen_uniform(seed + 1, n, 0, 1)


@pytest.mark.parametrize("dims,upper", [((1, 1), False), ((7, 9), True), ((64, 33), False), ((257, 129), True),
                                        ((1200, 900), False)])
def test_mprgp_iterations_on_the_device(ctx, dims, upper):
    # one row, a few, several rows a thread, and (1.08M rows: 2110 workgroups a product) sums finished by
    # their own kernel; with both bounds, expansion and proportioning steps of either sign
    A, b, lb = _obstacle(*dims, 3)
    ub = 0.02 + 0.1 * ua.gen_uniform(8, b.size, 0, 1) if upper else None
    q = ua.MPRGP(ctx, atol=1e-9, rtol=0, max_it=1000000)
    q.update(A)
    q.set_box_constraints(lb, ub)
    x, st = q.apply(b), q.status
    assert st["reason"] == 2 and st["gradient_norm"] <= 1e-9
    up = np.full(b.size, np.finfo(np.float64).max) if ub is None else ub
    assert np.all(x >= lb) and np.all(x <= up)
    # KKT: the projected gradient from an FP64 residual on the host; the loop's own g is a recurrence
    # whose rounding drift (its length times eps |A||x|) comes on top of atol
    g = A.to_scipy() @ x - b
    free = (x > lb) & (x < up)
    low, high = np.abs(x - lb) < 1e-14, np.abs(x - up) < 1e-14
    pg = np.where(free, g, 0.0) + np.where(low, np.minimum(g, 0), np.where(high, np.maximum(g, 0), 0.0))
    drift = st["iterates"] * 2.3e-16 * 16 * np.linalg.norm(x)
    assert np.linalg.norm(pg) <= 1e-9 + drift


@pytest.mark.parametrize("max_it", [1, 2, 17])
def test_mprgp_runs_the_same_in_one_call_and_step_by_step(ctx, max_it, capfd):
    A, b, lb = _obstacle(70, 41, 5)
    got = []
    for verbose in (0, 1):
        q = ua.MPRGP(ctx, atol=1e-30, rtol=0, max_it=max_it, verbose=verbose)
        q.update(A)
        q.set_box_constraints(lb, None)
        got.append((q.apply(b), q.status))
    assert np.array_equal(got[0][0], got[1][0])
    for key in ("iterates", "reason", "gradient_norm"):
        assert got[0][1][key] == got[1][1][key]
    assert got[0][1]["iterates"] == max_it and got[0][1]["reason"] == -5
    assert capfd.readouterr().out.count("\n") >= max_it


def test_mprgp_stops_on_negative_curvature(ctx):
    n = 200
    A = ua.Csr(np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.full(n, -1.0), (n, n))
    q = ua.MPRGP(ctx, atol=1e-9, rtol=0, max_it=50)
    q.update(A)
    q.set_box_constraints(np.full(n, -1e3), np.full(n, 1e3))
    x = q.apply(np.ones(n))
    assert np.all(x == 0) and q.status["iterates"] == 0


def _symmetric_random(n, per_row, seed):
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    M = sp.random(n, n, per_row / n, random_state=np.random.RandomState(seed), data_rvs=rng.standard_normal)
    M = (M + M.T).tocsr()
    d = np.asarray(abs(M).sum(axis=1)).ravel() + 1.0
    d[::17] = 0.0  # rows without a usable diagonal: d_inv = 0
    M.setdiag(d)
    return ua.Csr.from_scipy(M.tocsr())


@pytest.mark.parametrize("name", ["one", "nine", "nine_large", "ragged"])
@pytest.mark.parametrize("constrained,symmetric,add", [(1, 1, 1), (1, 0, 1), (0, 1, 0), (0, 0, 0), (1, 1, 0)])
@pytest.mark.parametrize("bounds", ["both", "lower"])
def test_colour_plan_sweep_equals_the_colours_one_by_one(ctx, name, constrained, symmetric, add, bounds):
    # slices that a colour does not fill, more than 16 entries a row (ragged: up to about 40), zero
    # diagonals, one row; a missing bound is the value that fills it
    A = {"one": lambda: ua.gen_stencil(ua.STENCIL_2D9, 1, 1, shift=1e-3),
         "nine": lambda: ua.gen_stencil(ua.STENCIL_2D9, 37, 23, shift=1e-3),
         "nine_large": lambda: ua.gen_stencil(ua.STENCIL_2D9, 301, 200, shift=1e-3),
         "ragged": lambda: _symmetric_random(700, 10, 3)}[name]()
    L, n = ua.lib(), A.shape[0]
    D = ua.DeviceCsr(ctx, A)
    color, rows = (ua.DeviceArray.from_numpy(ctx, np.zeros(n, np.int32)) for _ in range(2))
    nc = ctypes.c_int32()
    ua.check(L.uhip_graph_color(ctx.h, D.ref, 7, P(color), ctypes.byref(nc)))
    off = np.zeros(nc.value + 1, np.int32)
    ua.check(L.uhip_color_groups(ctx.h, n, P(color), nc, P(rows), ctypes.c_void_p(off.ctypes.data)))
    rng = np.random.default_rng(1)
    x0, b = rng.standard_normal(n), rng.standard_normal(n)
    lb = x0 - rng.uniform(0, 0.1, n)
    ub = x0 + rng.uniform(0, 0.1, n) if bounds == "both" else np.full(n, np.finfo(np.float64).max)
    dinv, x, bd, lbd, ubd = (ua.DeviceArray.from_numpy(ctx, v) for v in (np.zeros(n), x0, b, lb, ub))
    ua.check(L.uhip_pgs_dinv(ctx.h, D.ref, P(dinv)))
    r1, r2, c1, c2 = (ua.DeviceArray.from_numpy(ctx, np.full(n, 7.0)) for _ in range(4))
    D.residual(x, bd, r1)
    ua.check(L.uhip_vec_set_f64(ctx.h, n, 0.0, P(c1)))
    order = list(range(nc.value)) + (list(reversed(range(nc.value))) if symmetric else [])
    for k in order:
        ua.check(L.uhip_pgs_color_sweep(ctx.h, D.ref, int(off[k + 1] - off[k]),
                                        ctypes.c_void_p(rows.ptr + 4 * int(off[k])), P(dinv), P(r1), P(x), P(lbd), P(ubd),
                                        P(c1), constrained))
    plan = ctypes.c_void_p()
    ua.check(L.uhip_color_plan_create(ctx.h, D.ref, nc, P(rows), ctypes.c_void_p(off.ctypes.data), ctypes.byref(plan)))
    ua.check(L.uhip_spmv_residual_zero_f64(ctx.h, D.ref, P(x), P(bd), P(r2), P(c2)))
    assert np.array_equal(r1.numpy(), r2.numpy()) and np.all(c2.numpy() == 0)
    ua.check(L.uhip_color_plan_sweep(ctx.h, plan, P(dinv), P(r2), P(x), P(lbd), P(ubd) if bounds == "both" else None, P(c2),
                                     constrained, symmetric, add))
    assert np.array_equal(c1.numpy(), c2.numpy())
    assert np.array_equal(x.numpy(), x0 + c1.numpy() if add else x0)
    ua.check(L.uhip_color_plan_destroy(ctx.h, plan))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("rows", [1 << 18, (1 << 18) + 257, 1 << 19, (1 << 19) + 1, 255, 256, 257])
def test_dia_and_vi_products_where_the_rows_per_thread_change(ctx, dtype, rows):
    # 1D operators give any number of rows; 9 diagonals take the 16-bit masks (16 diagonals at once)
    import scipy.sparse as sp
    x = ua.gen_uniform(21, rows).astype(dtype)
    rng = np.random.default_rng(rows)
    for offsets in ((-1, 0, 1), (-40, -3, -2, -1, 0, 1, 2, 3, 40)):
        S = sp.diags([rng.standard_normal(rows).astype(np.float32)[:rows - abs(o)] for o in offsets], offsets)
        A = ua.Csr.from_scipy(S.tocsr())
        D = ua.DeviceCsr(ctx, A, dtype, fmt=ua.FMT_DIA)
        xd, yd = ua.DeviceArray.from_numpy(ctx, x), ua.DeviceArray(ctx, rows, dtype)
        D.spmv(xd, yd)
        ref = orc.spmv(A, x) if dtype == np.float64 else orc.spmv_f32(A, x)
        assert np.array_equal(yd.numpy(), ref)
    Pm = ua.gen_prolongation(rows, 1)
    D = ua.DeviceCsr(ctx, Pm, dtype, fmt=ua.FMT_VI)
    c = ua.gen_uniform(22, Pm.shape[1]).astype(dtype)
    cd, yd = ua.DeviceArray.from_numpy(ctx, c), ua.DeviceArray(ctx, rows, dtype)
    D.spmv(cd, yd)
    assert np.array_equal(yd.numpy(), orc.spmv(Pm, c) if dtype == np.float64 else orc.spmv_f32(Pm, c))


@pytest.mark.parametrize("ndiag,rows", [(27, 150000), (27, 150001), (27, 480000), (27, 480001), (16, 150001), (16, 480000),
                                        (16, 480001), (7, 480000), (7, 480001)])
def test_dia_product_and_its_dot_where_the_rows_per_thread_change(ctx, ndiag, rows):
    # with a dot the line lies lower for more than 16 diagonals; a sum of the dot takes 512 rows on either side
    import scipy.sparse as sp
    rng = np.random.default_rng(rows)
    offsets = np.arange(ndiag) - ndiag // 2
    A = ua.Csr.from_scipy(sp.diags([rng.standard_normal(rows - abs(o)) for o in offsets], offsets).tocsr())
    D = ua.DeviceCsr(ctx, A, fmt=ua.FMT_DIA)
    assert D.m.nparts == (rows + 511) // 512
    x = ua.gen_uniform(21, rows)
    xd, yd, zd, d = (ua.DeviceArray.from_numpy(ctx, v) for v in (x, 0 * x, 0 * x, np.zeros(1)))
    D.spmv(xd, yd)
    ua.check(ua.lib().uhip_spmv_dot(ctx.h, D.ref, P(xd), P(zd), P(d)))
    ref = orc.spmv(A, x)
    assert np.array_equal(yd.numpy(), ref) and np.array_equal(zd.numpy(), ref)
    assert abs(d.numpy()[0] - x @ ref) <= rows * 2.3e-16 * (np.abs(x) @ np.abs(ref))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("rows", [639999, 640000, 640001, 799999, 800000, 800001])
def test_vi_product_where_the_rows_per_lane_change(ctx, dtype, rows):
    Pm = ua.gen_prolongation(rows, 1)
    D = ua.DeviceCsr(ctx, Pm, dtype, fmt=ua.FMT_VI)
    c = ua.gen_uniform(22, Pm.shape[1]).astype(dtype)
    cd, yd = ua.DeviceArray.from_numpy(ctx, c), ua.DeviceArray(ctx, rows, dtype)
    D.spmv(cd, yd)
    assert np.array_equal(yd.numpy(), orc.spmv(Pm, c) if dtype == np.float64 else orc.spmv_f32(Pm, c))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("k", [1, 2, 4, 8, 16])
def test_products_with_several_columns_at_every_mean_row_length(ctx, dtype, k):
    # the mean decides how many entries are taken at once: rows shorter and longer than that, empty ones, and x with
    # values that are no numbers where no row has an entry (the row 0 that loads past a row's end fall on among them)
    rng = np.random.default_rng(k)
    code = ua.F64 if dtype == np.float64 else ua.F32
    for mean in list(range(1, 20)) + [27, 31]:
        n = 500
        lens = np.clip(mean + rng.integers(-3, 4, n), 0, None)
        lens[:n // 2] = mean
        lens[7] = 0
        rp = np.r_[0, np.cumsum(lens)].astype(np.int32)
        col = (1 + rng.integers(0, 400, rp[-1])).astype(np.int32)
        val = rng.standard_normal(rp[-1]).astype(dtype)
        X = rng.standard_normal((410, k)).astype(dtype)
        X[0] = X[401:] = np.nan
        D = ua.DeviceCsr(ctx, ua.Csr(rp, col, val, (n, 410)), dtype, block_nnz=1024)
        Xd, Yd = ua.DeviceArray.from_numpy(ctx, X.ravel()), ua.DeviceArray(ctx, n * k, dtype)
        ua.check(ua.lib().uhip_spmm(ctx.h, D.ref, k, P(Xd), code, P(Yd), code, 0, None, 0))
        got = Yd.numpy().reshape(n, k)
        want = np.zeros((n, k), dtype)
        for j in range(lens.max()):  # in entry order, the products rounded
            r = np.nonzero(lens > j)[0]
            want[r] = want[r] + val[rp[r] + j][:, None] * X[col[rp[r] + j]]
        assert np.array_equal(got, want), mean


@pytest.mark.parametrize("k", [1, 2, 4, 8, 16])
def test_batched_iteration_kernels_at_chunk_edges(ctx, k):
    # systems of 1 row, just about a workgroup's 256 rows and a chunk's 1024 rows, and several chunks. Dots of n
    # terms in another order differ by at most n eps sum |x||y| (n <= 2500: 6e-13 of it); the rest is exact.
    import scipy.sparse as sp
    L, P = ua.lib(), lambda a: ctypes.c_void_p(a.ptr) if a is not None else None
    sizes = [1, 255, 256, 257, 1023, 1024, 1025, 2500]
    seg = np.concatenate([[0], np.cumsum(sizes)])
    n, ns = int(seg[-1]), len(sizes)
    blocks = [sp.diags([ua.gen_uniform(5 + s, m).astype(np.float32) + 1 if o == 0 else -np.ones(max(m - abs(o), 0))
                        for o in (-3, -1, 0, 1, 3) if abs(o) < m], [o for o in (-3, -1, 0, 1, 3) if abs(o) < m])
              for s, m in enumerate(sizes)]
    A = ua.Csr.from_scipy(sp.block_diag(blocks).tocsr())
    r0, r1, c0 = [], [], [0]
    for s in range(ns):
        for a in range(seg[s], seg[s + 1], 1024):
            r0.append(a)
            r1.append(min(a + 1024, seg[s + 1]))
        c0.append(len(r0))
    rowseg = np.repeat(np.arange(ns), sizes)
    r0d, r1d, c0d, rsd = (ua.DeviceArray.from_numpy(ctx, np.asarray(v, np.int32)) for v in (r0, r1, c0, rowseg))
    up = lambda v: ua.DeviceArray.from_numpy(ctx, v)
    chunks = (len(r0), P(r0d), P(r1d))
    segs = (ns, P(c0d))

    def dots(x, y):
        t = x.astype(np.float64) * y.astype(np.float64)
        return (np.stack([t[seg[s]:seg[s + 1]].sum(axis=0) for s in range(ns)]),
                np.stack([np.abs(t[seg[s]:seg[s + 1]]).sum(axis=0) for s in range(ns)]) * 6e-13)

    X, Rv, x0 = (ua.gen_normal(60 + i, n * k).reshape(n, k) for i in range(3))
    D = ua.DeviceCsr(ctx, A)
    Xd, Yd, out = up(X), ua.DeviceArray(ctx, n * k), ua.DeviceArray(ctx, ns * k)
    ua.check(L.uhip_spmm_dot(ctx.h, D.ref, k, P(Xd), P(Yd), *chunks, *segs, P(out)))
    Y = np.stack([orc.spmv(A, np.ascontiguousarray(X[:, j])) for j in range(k)], axis=1)
    assert np.array_equal(Yd.numpy().reshape(n, k), Y)
    ref, tol = dots(X, Y)
    assert np.all(np.abs(out.numpy().reshape(ns, k) - ref) <= tol)

    # r -= alpha Ap, its copy and |r|; a step of 0 leaves r as it is
    alpha, beta = (ua.gen_normal(70 + i, ns * k).reshape(ns, k) for i in range(2))
    alpha[1] = 0
    ad, bd, Rd, R32 = up(alpha), up(beta), up(Rv), ua.DeviceArray(ctx, n * k, np.float32)
    ua.check(L.uhip_bcg_residual(ctx.h, k, P(rsd), P(ad), P(Rd), P(Yd), P(R32), *chunks, *segs, P(out)))
    Rn = Rv - alpha[rowseg] * Y
    assert np.array_equal(Rd.numpy().reshape(n, k), Rn)
    assert np.array_equal(R32.numpy().reshape(n, k), Rn.astype(np.float32))
    ref, tol = dots(Rn, Rn)
    assert np.all(np.abs(out.numpy().reshape(ns, k) ** 2 - ref) <= tol + 1e-15 * ref)

    # last smoothing step: the bits of the step without a dot
    coef = up(ua.gen_normal(80, 3 * ns))
    for dt, code in ((np.float64, ua.F64), (np.float32, ua.F32)):
        Dt = ua.DeviceCsr(ctx, A, dtype=dt)
        pd, xd, o1, o2 = up(X.astype(dt)), up(x0.astype(dt)), ua.DeviceArray(ctx, n * k, dt), ua.DeviceArray(ctx, n * k, dt)
        ua.check(L.uhip_spmm_cheb_step(ctx.h, Dt.ref, k, P(pd), code, None, P(xd), P(o1), code, P(o1), P(o1), P(rsd), P(coef), 1))
        ua.check(L.uhip_spmm_cheb_last_dot(ctx.h, Dt.ref, k, P(pd), None, P(xd), P(o2), P(rsd), P(coef), P(Rd), *chunks, *segs,
                                           P(out)))
        Z = o2.numpy().reshape(n, k)
        assert np.array_equal(o1.numpy().reshape(n, k), Z)
        ref, tol = dots(Z, Rn)
        assert np.all(np.abs(out.numpy().reshape(ns, k) - ref) <= tol)
        # x += alpha p while the iteration runs, p = z + beta p while pairs are active
        for pending, active in ((0, 1), (1, 0), (1, 1)):
            xs, ps, pe, ac = up(x0), up(X), up(np.array([pending], np.int32)), up(np.array([active], np.int32))
            ua.check(L.uhip_bcg_xpupdate(ctx.h, n, k, P(rsd), P(ad), P(bd), P(xs), P(ps), P(o2), code, P(pe), P(ac)))
            assert np.array_equal(xs.numpy().reshape(n, k), x0 + alpha[rowseg] * X if pending else x0)
            assert np.array_equal(ps.numpy().reshape(n, k),
                                  Z.astype(np.float64) + beta[rowseg] * X if pending and active else X)


def _hub(n, length):
    """-1 / 4 chains with one row (and column) of `length` entries: its slice of 64 rows is 64 * length wide."""
    import scipy.sparse as sp
    S = sp.diags([-1.0, 4.0, -1.0], [-1, 0, 1], shape=(n, n)).tolil()
    S[n // 2, 1:1 + length] = -1e-4
    S[1:1 + length, n // 2] = -1e-4
    S[n // 2, n // 2] = 4.0
    S = S.tocsr()
    S.sort_indices()
    return ua.Csr.from_scipy(S)


@pytest.mark.parametrize("length,status", [(20000, 0), (60000, -5)])
@pytest.mark.parametrize("bounds", [None, "lower", "both"])
def test_gauss_seidel_with_a_row_too_long_for_the_colour_plan(ctx, length, status, bounds):
    # the plan holds up to 4 nnz + 2^20 slots: 64 * 20,000 among 340,000 entries fit, 64 * 60,000 do not and the
    # sweeps run from the matrix. The steps of the solver, colour by colour from the matrix, bit for bit
    n, steps = 100000, 2
    A = _hub(n, length)
    L = ua.lib()
    D = ua.DeviceCsr(ctx, A)
    color, rows = (ua.DeviceArray.from_numpy(ctx, np.zeros(n, np.int32)) for _ in range(2))
    nc, plan = ctypes.c_int32(), ctypes.c_void_p()
    ua.check(L.uhip_graph_color(ctx.h, D.ref, 0x5eed, P(color), ctypes.byref(nc)))
    off = np.zeros(nc.value + 1, np.int32)
    ua.check(L.uhip_color_groups(ctx.h, n, P(color), nc, P(rows), ctypes.c_void_p(off.ctypes.data)))
    st = L.uhip_color_plan_create(ctx.h, D.ref, nc, P(rows), ctypes.c_void_p(off.ctypes.data), ctypes.byref(plan))
    assert st == status
    if st == 0:
        ua.check(L.uhip_color_plan_destroy(ctx.h, plan))
    b = ua.gen_uniform(3, n)
    lb, ub = np.full(n, -0.2), np.full(n, 0.3 if bounds == "both" else np.finfo(np.float64).max)
    dinv, x, r, c, bd, lbd, ubd = (ua.DeviceArray.from_numpy(ctx, v) for v in (np.zeros(n),) * 4 + (b, lb, ub))
    ua.check(L.uhip_pgs_dinv(ctx.h, D.ref, P(dinv)))
    for _ in range(steps):
        D.residual(x, bd, r)
        ua.check(L.uhip_vec_set_f64(ctx.h, n, 0.0, P(c)))
        for k in list(range(nc.value)) + list(reversed(range(nc.value))):
            ua.check(L.uhip_pgs_color_sweep(ctx.h, D.ref, int(off[k + 1] - off[k]),
                                            ctypes.c_void_p(rows.ptr + 4 * int(off[k])), P(dinv), P(r), P(x), P(lbd),
                                            P(ubd), P(c), 0 if bounds is None else 1))
        ua.check(L.uhip_vec_axpy_f64(ctx.h, n, 1.0, P(c), P(x)))
    # the check that ends the loop comes after the first step and every check_s_norm_each ones
    q = ua.ProjectedGaussSeidel(ctx, stol=0.0, max_it=steps - 1, check_s_norm_each=steps - 1)
    q.update(A)
    if bounds:
        q.set_box_constraints(lb, ub if bounds == "both" else None)
    assert np.array_equal(q.apply(b), x.numpy())


def test_colour_plan_of_more_slots_than_32_bits_count(ctx):
    # 2^20 rows of one colour, one of 4,096 (+ 1 in the first slice) entries in every 64: 2^32 + 64 slots, which 32
    # bits take for 64. Refused before anything is filled
    n, length = 1 << 20, 4096
    lens = np.ones(n, np.int64)
    lens[::64] = length
    lens[0] += 1
    rp = np.concatenate([[0], np.cumsum(lens)])
    start = np.repeat(np.arange(n) % (n - length - 1), lens)
    col = (start + np.arange(rp[-1]) - np.repeat(rp[:-1], lens)).astype(np.int32)
    A = ua.Csr(rp.astype(np.int32), col, np.ones(rp[-1]), (n, n))
    assert int(sum(64 * lens.reshape(-1, 64).max(axis=1))) == (1 << 32) + 64
    D = ua.DeviceCsr(ctx, A, block_nnz=2048)
    rows, off, plan = ua.DeviceArray.from_numpy(ctx, np.arange(n, dtype=np.int32)), np.array([0, n], np.int32), ctypes.c_void_p()
    assert ua.lib().uhip_color_plan_create(ctx.h, D.ref, 1, P(rows), ctypes.c_void_p(off.ctypes.data), ctypes.byref(plan)) == -5
    assert not plan.value


@pytest.mark.parametrize("n", [1, 255, 1025, 70001])
@pytest.mark.parametrize("z_dtype", [np.float64, np.float32])
@pytest.mark.parametrize("deferred", [False, True])
def test_cg_update_with_its_dot_finished_or_left_as_partial_sums(ctx, n, z_dtype, deferred):
    # x += alpha p, p = z + (z.r / rz) p by uhip_cg_xpupdate3, one entry a thread and several workgroups, with z.r as
    # uhip_vec_dots left it; s[i_num] holds z.r afterwards either way, and alpha and |r| are reported
    L, rng = ua.lib(), np.random.default_rng(n)
    x, p, z, r = (rng.standard_normal(n) for _ in range(4))
    z = z.astype(z_dtype)
    parts = ua.DeviceArray.from_numpy(ctx, np.r_[4.0, np.zeros(L.uhip_cg_residual_parts(n) - 1)])
    s = ua.DeviceArray.from_numpy(ctx, np.array([2.0, 0.0, 0.5, -1.0, 0.0]))  # rz, p.Ap, alpha, -, z.r
    xd, pd, zd, rd, z64 = (ua.DeviceArray.from_numpy(ctx, v) for v in (x, p, z, r, z.astype(np.float64)))
    slot = ctypes.c_void_p(s.ptr + 32)
    ua.check(L.uhip_cg_begin(ctx.h))
    if deferred:
        ua.check(L.uhip_ctx_defer_sum(ctx.h, slot, 4096))
    one = (ctypes.c_void_p * 1)
    ua.check(L.uhip_vec_dots_f64(ctx.h, n, 1, one(z64.ptr), one(rd.ptr), slot))
    ua.check(L.uhip_cg_xpupdate3(ctx.h, n, P(xd), P(pd), P(zd), ua.F32 if z_dtype == np.float32 else ua.F64, P(s), 2, 4, 0,
                                 P(parts), 1))
    alpha, norm = ctypes.c_double(), ctypes.c_double()
    ua.check(L.uhip_cg_wait(ctx.h, 1, ctypes.byref(alpha), ctypes.byref(norm)))
    ua.check(L.uhip_ctx_defer_sum(ctx.h, None, 0))
    assert (alpha.value, norm.value) == (0.5, 2.0)
    got, eps = s.numpy(), 2.3e-16
    num, den = float(z.astype(np.float64) @ r), float(np.abs(z.astype(np.float64)) @ np.abs(r))
    assert abs(got[4] - num) <= n * eps * den and np.array_equal(got[:4], [2.0, 0.0, 0.5, -1.0])
    assert np.array_equal(xd.numpy(), x + 0.5 * p)
    assert np.array_equal(pd.numpy(), z.astype(np.float64) + (got[4] / 2.0) * p)


@pytest.mark.parametrize("between", ["nothing", "dot elsewhere", "reduction", "read", "other consumer", "switched off"])
def test_a_dot_left_as_partial_sums_is_finished_ahead_of_other_work(ctx, between):
    n = 50001
    L, rng = ua.lib(), np.random.default_rng(5)
    x, p, z, r, w = (rng.standard_normal(n) for _ in range(5))
    s = ua.DeviceArray.from_numpy(ctx, np.array([2.0, 1.0, 0.5, 3.0, -7.0, 0.0]))
    xd, pd, zd, rd, wd = (ua.DeviceArray.from_numpy(ctx, v) for v in (x, p, z, r, w))
    parts = ua.DeviceArray.from_numpy(ctx, np.zeros(L.uhip_cg_residual_parts(n)))
    slot, other, one = ctypes.c_void_p(s.ptr + 32), ctypes.c_void_p(s.ptr + 40), (ctypes.c_void_p * 1)
    ua.check(L.uhip_cg_begin(ctx.h))
    ua.check(L.uhip_ctx_defer_sum(ctx.h, slot, 4096))
    ua.check(L.uhip_vec_dots_f64(ctx.h, n, 1, one(zd.ptr), one(rd.ptr), slot))
    num, bound = float(z @ r), n * 2.3e-16 * float(np.abs(z) @ np.abs(r))
    if between == "dot elsewhere":
        ua.check(L.uhip_vec_dots_f64(ctx.h, n, 1, one(wd.ptr), one(wd.ptr), other))
    elif between == "reduction":
        ua.check(L.uhip_vec_reduce_f64(ctx.h, n, P(wd), 3, other))
    elif between == "read":
        h = np.zeros(1)
        ua.check(L.uhip_read_scalars(ctx.h, slot, 1, ctypes.c_void_p(h.ctypes.data)))
        assert abs(h[0] - num) <= bound
    elif between == "other consumer":  # it does not ask for this slot: s[1] is finished already
        q = ua.DeviceArray.from_numpy(ctx, np.zeros(n))
        ua.check(L.uhip_cg_residual2_f64(ctx.h, n, P(rd), P(wd), P(q), None, P(s), 0, 1, 3, P(parts)))
    elif between == "switched off":
        ua.check(L.uhip_ctx_defer_sum(ctx.h, None, 0))
    ua.check(L.uhip_cg_xpupdate3(ctx.h, n, P(xd), P(pd), P(zd), ua.F64, P(s), 2, 4, 0, P(parts), 1))
    ua.check(L.uhip_ctx_defer_sum(ctx.h, None, 0))
    got = s.numpy()
    assert abs(got[4] - num) <= bound
    assert np.array_equal(pd.numpy(), z + (got[4] / 2.0) * p) and np.array_equal(xd.numpy(), x + 0.5 * p)


def test_only_the_next_dot_to_a_slot_may_be_left_as_partial_sums(ctx):
    n = 5000
    L = ua.lib()
    v, s = ua.DeviceArray.from_numpy(ctx, np.ones(n)), ua.DeviceArray.from_numpy(ctx, np.zeros(4))
    one = (ctypes.c_void_p * 1)
    ua.check(L.uhip_ctx_defer_sum(ctx.h, P(s), 4096))
    for _ in range(2):
        ua.check(L.uhip_vec_dots_f64(ctx.h, n, 1, one(v.ptr), one(v.ptr), P(s)))
    h = s.numpy()  # a copy of memory, which finishes nothing
    ua.check(L.uhip_ctx_defer_sum(ctx.h, None, 0))
    assert h[0] == n


@pytest.mark.parametrize("n", [4096 * 512, 4096 * 512 + 1])
def test_cg_loop_where_its_dots_stop_being_left_as_partial_sums(ctx, n):
    # a DIA product of 4096 partial sums (2^21 rows, the loop's lines for both dots) and of 4097: three iterations with
    # the dots left where few enough, and with the finished ones of uhip_cg_residual_f64 and uhip_cg_xpupdate2
    L = ua.lib()
    rp = np.r_[0, np.cumsum(np.r_[2, np.full(n - 2, 3), 2])].astype(np.int32)
    col = np.empty(rp[-1], np.int32)
    row = np.repeat(np.arange(n, dtype=np.int32), np.diff(rp))
    col[:] = row + (np.arange(rp[-1]) - rp[row]) - 1
    col[:2] += 1
    A = ua.Csr(rp, col, np.where(row == col, 2.5, -1.0), (n, n))
    D = ua.DeviceCsr(ctx, A, fmt=ua.FMT_DIA)
    assert D.m.nparts == (n + 511) // 512
    b = ua.gen_uniform(3, n)
    most, z_most, one = 4096, 4096 if n <= 1 << 21 else 0, (ctypes.c_void_p * 1)
    RZ, PAP, ALPHA, NORM, RZNEW = range(5)
    out = []
    for left in (True, False):
        dinv, r, p = (ua.DeviceArray.from_numpy(ctx, v) for v in (np.full(n, 0.4), b, 0.4 * b))
        x, Ap, rn, z = (ua.DeviceArray.from_numpy(ctx, np.zeros(n)) for _ in range(4))
        s = ua.DeviceArray.from_numpy(ctx, np.r_[0.4 * (b @ b), np.zeros(7)])
        at = lambda i: ctypes.c_void_p(s.ptr + 8 * i)
        parts = ua.DeviceArray.from_numpy(ctx, np.zeros(L.uhip_cg_residual_parts(n)))
        ua.check(L.uhip_cg_begin(ctx.h))
        rz, rznew, norms = RZ, RZNEW, []
        for seq in range(1, 4):
            if left:
                ua.check(L.uhip_ctx_defer_sum(ctx.h, at(PAP), most))
            ua.check(L.uhip_spmv_dot(ctx.h, D.ref, P(p), P(Ap), at(PAP)))
            if left:
                ua.check(L.uhip_cg_residual2_f64(ctx.h, n, P(r), P(Ap), P(rn), None, P(s), rz, PAP, ALPHA, P(parts)))
                ua.check(L.uhip_ctx_defer_sum(ctx.h, at(rznew), z_most))
            else:
                ua.check(L.uhip_cg_residual_f64(ctx.h, n, P(r), P(Ap), P(rn), None, P(s), rz, PAP, ALPHA, NORM))
            ua.check(L.uhip_vec_emul_f64(ctx.h, n, P(dinv), P(rn), P(z)))
            ua.check(L.uhip_vec_dots_f64(ctx.h, n, 1, one(z.ptr), one(rn.ptr), at(rznew)))
            if left:
                ua.check(L.uhip_cg_xpupdate3(ctx.h, n, P(x), P(p), P(z), ua.F64, P(s), ALPHA, rznew, rz, P(parts), seq))
                a, norm = ctypes.c_double(), ctypes.c_double()
                ua.check(L.uhip_cg_wait(ctx.h, seq, ctypes.byref(a), ctypes.byref(norm)))
                norms.append(norm.value)
            else:
                ua.check(L.uhip_cg_xpupdate2(ctx.h, n, P(x), P(p), P(z), ua.F64, P(s), ALPHA, rznew, rz))
                norms.append(s.numpy()[NORM])
            r, rn, rz, rznew = rn, r, rznew, rz
        ua.check(L.uhip_ctx_defer_sum(ctx.h, None, 0))
        out.append((x.numpy(), r.numpy(), p.numpy(), np.array(norms)))
    # the same sums of n terms added in another order: n eps of their terms' size, through three steps
    for u, v in zip(*out):
        assert np.linalg.norm(u - v) <= 3 * n * 2.3e-16 * np.linalg.norm(v)
    rr = b - A.to_scipy() @ out[0][0]
    assert abs(np.linalg.norm(rr) - out[0][3][-1]) <= 1e-12 * np.linalg.norm(b)


@pytest.mark.parametrize("nx", [128, 129])
def test_multigrid_cg_on_both_sides_of_two_to_the_21_rows(ctx, nx):
    A = ua.gen_stencil(ua.STENCIL_3D7, nx, 128, 128)
    b = ua.gen_uniform(1, A.shape[0])
    atol = 1e-8 * np.linalg.norm(b)
    ua.srand(1)
    cg = ua.ConjugateGradient(ctx, "multigrid", atol=atol, rtol=1e-30, stol=1e-30, max_it=40, pre_smoothing_steps=2,
                              post_smoothing_steps=2)
    cg.set_transfer_operators(ua.mg_hierarchy(nx, 128, 128, 5))
    x = cg.solve(A, b)
    st = cg.status
    assert st["reason"] == 2 and st["iterates"] <= 20
    res = np.linalg.norm(b - A.to_scipy() @ x)
    # the recurrence's residual moves from the true one by eps |A| |x| an iteration (|A| <= 12)
    assert abs(res - st["gradient_norm"]) <= 20 * 12 * 2.3e-16 * np.linalg.norm(x) and st["gradient_norm"] <= atol


def test_loops_inside_loops_are_counted(ctx):
    L = ua.lib()
    for _ in range(7):
        ua.check(L.uhip_ctx_enter_loop(ctx.h))
    assert L.uhip_ctx_enter_loop(ctx.h) == -5
    for _ in range(7):
        ua.check(L.uhip_ctx_leave_loop(ctx.h))
    assert L.uhip_ctx_leave_loop(ctx.h) == -1


def test_setup_functions_of_several_threads_on_one_context(ctx):
    # products and transposes (whose sizes come back through the context) beside dots read back by another thread:
    # everything runs on the one stream, in some order
    import threading
    L = ua.lib()
    mats = [(_rows_of_lengths([7] * n, n, n), _rows_of_lengths([5] * n, m, m)) for n, m in ((300, 400), (1500, 90))]
    dev = [(ua.DeviceCsr(ctx, A), ua.DeviceCsr(ctx, B)) for A, B in mats]
    want = [orc.spgemm(A, B) for A, B in mats]
    v, s = ua.DeviceArray.from_numpy(ctx, np.ones(5000)), ua.DeviceArray.from_numpy(ctx, np.zeros(1))
    wrong, done = [], threading.Event()

    def products(k):
        for _ in range(60):
            C, T = ua.uhip_csr(), ua.uhip_csr()
            ua.check(L.uhip_csr_spgemm(ctx.h, dev[k][0].ref, dev[k][1].ref, ctypes.byref(C)))
            ua.check(L.uhip_csr_transpose(ctx.h, ctypes.byref(C), ctypes.byref(T)))
            if C.nnz != want[k][1].size or T.nnz != C.nnz or T.nrows != C.ncols:
                wrong.append((k, C.nnz, T.nnz))
            ua.check(L.uhip_csr_free(ctx.h, ctypes.byref(T)))
            if not np.array_equal(_csr_of(ctx, C).val, want[k][2]):
                wrong.append((k, "values"))

    def dots():
        one, h = (ctypes.c_void_p * 1), np.zeros(1)
        while not done.is_set():
            ua.check(L.uhip_vec_dots_f64(ctx.h, v.n, 1, one(v.ptr), one(v.ptr), P(s)))
            ua.check(L.uhip_read_scalars(ctx.h, P(s), 1, ctypes.c_void_p(h.ctypes.data)))
            if h[0] != v.n:
                wrong.append(("dot", h[0]))

    threads = [threading.Thread(target=products, args=(k,)) for k in (0, 1)]
    reader = threading.Thread(target=dots)
    for t in threads + [reader]:
        t.start()
    for t in threads:
        t.join(60)
    done.set()
    reader.join(60)
    assert not wrong and not any(t.is_alive() for t in threads + [reader])


# A launch may have less than 2^32 threads: the kernels with several lanes a row get there at 2^27 rows and more.

def _unplanned(nrows, ncols, rowptr, col, val):
    A = ua.uhip_csr()
    A.nrows, A.ncols, A.nnz, A.dtype = nrows, ncols, val.n, ua.F64
    A.rowptr, A.col, A.val = rowptr.ptr, col.ptr, val.ptr
    return A


def test_transpose_of_more_columns_than_a_launch_of_32_lanes_each(ctx):
    m = (1 << 27) + 9
    cols = [[0, 5, m - 10], [5, (1 << 26) + 1, m - 9, m - 1], [m - 1]]
    col = np.concatenate(cols).astype(np.int32)
    val = np.arange(1.0, col.size + 1)
    A = ua.Csr(np.array([0, 3, 7, 8], np.int32), col, val, (3, m))
    D, T = ua.DeviceCsr(ctx, A, block_nnz=1024), ua.uhip_csr()
    ua.check(ua.lib().uhip_csr_transpose(ctx.h, D.ref, ctypes.byref(T)))
    got = _csr_of(ctx, T)
    want = np.zeros(m + 1, np.int32)
    for c in np.unique(col):
        want[c + 1:] += np.count_nonzero(col == c)
    order = np.argsort(col, kind="stable")
    assert got.shape == (m, 3) and np.array_equal(got.rowptr, want)
    assert np.array_equal(got.val, val[order]) and np.array_equal(got.col, np.repeat([0, 1, 2], [3, 4, 1])[order])


def test_spgemm_of_more_rows_than_a_launch_of_32_lanes_each(ctx):
    n = (1 << 27) + 5
    B = _rows_of_lengths([20, 24], 60, 3)  # 22 entries a row on average: 32 lanes a row of the product
    rows = np.array([0, 1, (1 << 25) + 3, (1 << 26) - 1, (1 << 27) - 1, 1 << 27, n - 2, n - 1])
    rp = np.zeros(n + 1, np.int32)
    for r in rows:
        rp[r + 1:] += 2
    small = ua.Csr(np.arange(0, 2 * rows.size + 1, 2, dtype=np.int32), np.tile([0, 1], rows.size).astype(np.int32),
                   np.arange(1.0, 2 * rows.size + 1), (rows.size, 2))
    A = _unplanned(n, 2, rpd := ua.DeviceArray.from_numpy(ctx, rp), col := ua.DeviceArray.from_numpy(ctx, small.col),
                   val := ua.DeviceArray.from_numpy(ctx, small.val))
    DB, C = ua.DeviceCsr(ctx, B), ua.uhip_csr()
    ua.check(ua.lib().uhip_csr_spgemm(ctx.h, ctypes.byref(A), DB.ref, ctypes.byref(C)))
    got = _csr_of(ctx, C)
    del rpd, col, val
    srp, scol, sval, _ = orc.spgemm(small, B)
    want = np.zeros(n + 1, np.int32)
    for r, k in zip(rows, np.diff(srp)):
        want[r + 1:] += k
    assert got.shape == (n, 60) and np.array_equal(got.rowptr, want)
    assert np.array_equal(got.col, scol) and np.array_equal(got.val, sval)


def test_product_with_16_columns_of_more_rows_than_a_launch_of_8_lanes_each(ctx):
    k, n = 16, (1 << 29) + 3  # 69 GB of results
    L = ua.lib()
    rows = np.array([0, 7, (1 << 28) + 1, (1 << 28) + 2, (1 << 29) - 1, 1 << 29, n - 1])
    rp = np.zeros(n + 1, np.int32)
    for i, r in enumerate(rows):
        rp[r + 1:] = i + 1
    rpd, col, val = (ua.DeviceArray.from_numpy(ctx, v) for v in (rp, np.arange(rows.size, dtype=np.int32) % 3,
                                                                 np.arange(1.0, rows.size + 1)))
    del rp
    A = _unplanned(n, 3, rpd, col, val)
    X = np.arange(3.0 * k).reshape(3, k) + 1
    Xd, Y = ua.DeviceArray.from_numpy(ctx, X.ravel()), ua.DeviceArray(ctx, n * k)
    ua.check(L.uhip_spmm(ctx.h, ctypes.byref(A), k, P(Xd), ua.F64, P(Y), ua.F64, 0, None, 0))
    got = np.zeros(k)
    for r, want in list(zip(rows, [(i + 1.0) * X[i % 3] for i in range(rows.size)])) + [(n - 2, 0 * X[0]), (1 << 27, 0 * X[0])]:
        ua.check(L.uhip_memcpy_dtoh(ctx.h, ctypes.c_void_p(got.ctypes.data), ctypes.c_void_p(Y.ptr + 8 * k * int(r)), got.nbytes))
        assert np.array_equal(got, want), r


# The single steps of the loops that now decide on the device or fuse them: entries of the C ABI on their own.

def _free(x, g, lb, ub):
    return np.where((lb < x) & (x < ub), g, 0.0)


@pytest.mark.parametrize("n", [1, 255, 1025, 70001])
def test_mprgp_steps_one_by_one(ctx, n):
    L, rng, s = ua.lib(), np.random.default_rng(n), ctx.scalars
    lb, ub = np.full(n, -0.1), np.full(n, 0.25)
    x = np.clip(rng.uniform(-0.2, 0.35, n), lb, ub)
    g, p, Ap = (rng.standard_normal(n) for _ in range(3))
    up = lambda v: ua.DeviceArray.from_numpy(ctx, v)
    xd, gd, pd, Apd, lbd, ubd = map(up, (x, g, p, Ap, lb, ub))
    at = ctypes.c_void_p(s + 8 * 40)
    ua.check(L.uhip_mprgp_alpha_f_f64(ctx.h, n, P(xd), P(pd), P(lbd), P(ubd), at))
    with np.errstate(divide="ignore", invalid="ignore"):
        want = min(np.where(p > 0, (x - lb) / p, 1e15).min(), np.where(p < 0, (x - ub) / p, 1e15).min())
    assert ctx.read_scalars(s + 8 * 40, 1)[0] == want

    x2 = up(x)
    ua.check(L.uhip_mprgp_expand_f64(ctx.h, n, P(x2), P(gd), P(pd), P(Apd), P(lbd), P(ubd), 0.3, 0.7))
    xi, gi = x - 0.3 * p, g - 0.3 * Ap
    assert np.array_equal(x2.numpy(), np.clip(xi - 0.7 * _free(xi, gi, lb, ub), lb, ub))

    x3, g3, p3 = up(x), up(g), up(p)
    ua.check(L.uhip_mprgp_proportion_f64(ctx.h, n, P(x3), P(g3), P(pd), P(Apd), P(lbd), P(ubd), P(p3), 0.2))
    xi, gi = x - 0.2 * p, g - 0.2 * Ap
    assert np.array_equal(x3.numpy(), xi) and np.array_equal(g3.numpy(), gi)
    assert np.array_equal(p3.numpy(), _free(xi, gi, lb, ub))

    f = ua.DeviceArray(ctx, n)
    ua.check(L.uhip_mprgp_free_grad_f64(ctx.h, n, P(xd), P(gd), P(lbd), P(ubd), P(f)))
    assert np.array_equal(f.numpy(), _free(x, g, lb, ub))

    sc, p4 = up(np.array([3.0, 4.0])), up(p)
    ua.check(L.uhip_mprgp_pupdate_f64(ctx.h, n, P(p4), P(gd), P(sc), 0, 1))
    assert np.array_equal(p4.numpy(), g - 0.75 * p)


@pytest.mark.parametrize("slot", [0, 1])
def test_scalars_read_back_while_the_stream_goes_on(ctx, slot):
    L = ua.lib()
    v = ua.DeviceArray.from_numpy(ctx, np.array([1.0, 2.0, 3.0, 4.0]))
    ua.check(L.uhip_fetch_scalars(ctx.h, slot, P(v), 3))
    ua.check(L.uhip_vec_scale_f64(ctx.h, 4, 2.0, P(v)))  # enqueued after the copy
    h = np.zeros(3)
    ua.check(L.uhip_fetch_wait(ctx.h, slot, 3, ctypes.c_void_p(h.ctypes.data)))
    assert np.array_equal(h, [1, 2, 3]) and np.array_equal(v.numpy(), [2, 4, 6, 8])
    assert L.uhip_fetch_scalars(ctx.h, 2, P(v), 3) == -1


@pytest.mark.parametrize("k", [1, 2, 4, 8, 16])
def test_batched_cg_stages_one_by_one(ctx, k):
    L, rng = ua.lib(), np.random.default_rng(k)
    sizes = [1, 255, 300]
    n, ns, m = sum(sizes), len(sizes), len(sizes) * k
    rowseg = np.repeat(np.arange(ns), sizes).astype(np.int32)
    up = lambda v: ua.DeviceArray.from_numpy(ctx, v)
    x, p, r, Ap, z = (rng.standard_normal((n, k)) for _ in range(5))
    rz, pap, rznew = (rng.uniform(1, 2, m) for _ in range(3))
    pap[0] = 0.0                     # alpha is not finite: that pair stops
    flags = np.zeros(m, np.int32)
    flags[m - 1] = 1                 # a pair that has converged
    xd, pd, rd, Apd, zd, rsd, fl = map(up, (x, p, r, Ap, z, rowseg, flags))
    st = [up(v) for v in (rz, pap, np.zeros(m), np.zeros(m), rznew, np.zeros(m), np.zeros(m))]
    state = (ctypes.c_void_p * 7)(*[v.ptr for v in st])
    conv, it, act = (up(np.zeros(q, np.int32)) for q in (m, 1, 1))

    def step(stage):
        ua.check(L.uhip_bcg_step(ctx.h, stage, n, k, m, P(rsd), P(xd), P(pd), P(rd), P(Apd), P(zd), state, P(fl), P(conv),
                                 P(it), P(act)))

    step(0)
    with np.errstate(divide="ignore"):
        alpha = np.where((flags != 0) | (pap == 0), 0.0, rz / pap)
    a = alpha.reshape(ns, k)[rowseg]
    assert np.array_equal(st[2].numpy(), alpha) and fl.numpy()[0] == (2 if m > 1 else 1)
    assert np.array_equal(xd.numpy().reshape(n, k), x + a * p) and np.array_equal(rd.numpy().reshape(n, k), r - a * Ap)
    step(2)
    beta = np.where(fl.numpy() != 0, 0.0, rznew / rz)
    assert np.array_equal(st[3].numpy(), beta) and np.array_equal(st[0].numpy(), rznew)
    assert np.array_equal(pd.numpy().reshape(n, k), z + beta.reshape(ns, k)[rowseg] * p)
    assert L.uhip_bcg_step(ctx.h, 3, n, k, m, P(rsd), P(xd), P(pd), P(rd), P(Apd), P(zd), state, P(fl), P(conv), P(it),
                           P(act)) == -1
