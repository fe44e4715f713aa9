"""Grouped block factorisations through the C ABI at the sizes where their kernels change course
(needs an MI355X).

Householder QR (xh_block_qr): rows around the 64, 128, 192, 256 and 1024 that pick the
kernel, single rows and columns, more columns than one panel, wide blocks, dependent columns,
reflectors or working copies too large for LDS, and a middle dimension above min(m, n).  Bounds (Higham, Accuracy and Stability of Numerical Algorithms, 2nd
ed., theorem 19.4): ||A - Q R||_F and ||Q^T Q - I||_F are at most about m n eps times ||A||_F and
sqrt(n); the tests allow m n eps with the constant 1, which random rounding stays far below.
"""
import ctypes as C

import numpy as np
import pytest

from xped_amd import _lib
from xped_amd._lib import lib

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _run(rt, fn, blocks, out_sizes, items):
    """Uploads the blocks (column-major), calls fn(items, n, dA, *outs) and downloads the outputs."""
    L, ctx = lib(), rt.ctx()
    flat = np.concatenate([b.T.reshape(-1) for b in blocks])
    dA, outs = C.c_void_p(), [C.c_void_p() for _ in out_sizes]
    for p, n in zip([dA] + outs, [flat.size] + list(out_sizes)):
        assert L.xh_alloc(ctx, 8 * max(n, 1), C.byref(p)) == 0
    L.xh_upload(ctx, dA, flat.ctypes.data, 8 * flat.size)
    arr = (_lib.xh_factor_item * len(items))(*items)
    assert fn(ctx, arr, len(items), dA, *outs) == 0, L.xh_last_error(ctx)
    res = []
    for p, n in zip(outs, out_sizes):
        x = np.empty(n)
        L.xh_download(ctx, x.ctypes.data, p, 8 * n)
        res.append(x)
    for p in [dA] + outs:
        L.xh_free(ctx, p)
    return res


QR_SHAPES = [(1, 1), (1, 7), (7, 1), (16, 16), (17, 16), (64, 64), (65, 33), (63, 5), (128, 100), (129, 40), (256, 70), (257, 60), (1024, 15),
             (1025, 15), (20, 300), (190, 180), (130, 300), (192, 90), (193, 66), (256, 250), (700, 200), (2000, 40), (48, 700)]


def test_block_qr_across_kernel_edges(rt):
    r = np.random.default_rng(5)
    blocks = [r.uniform(-1, 1, s) for s in QR_SHAPES]
    dep = r.uniform(-1, 1, (40, 12))
    dep[:, 3] = 0.0  # no reflector: tau = 0
    dep[:, 7] = 2.0 * dep[:, 1]
    blocks.append(dep)
    blocks.append(np.eye(33))
    mids = [min(b.shape) for b in blocks]
    mids[4], mids[3] = 19, 16  # a middle dimension above the block's rows: zero columns of Q, zero rows of R
    items, ao, uo, vo = [], 0, 0, 0
    for b, k in zip(blocks, mids):
        m, n = b.shape
        items.append(_lib.xh_factor_item(ao, uo, k, vo, m, n))
        ao, uo, vo = ao + m * n, uo + m * k, vo + k * n
    Q, R = _run(rt, lib().xh_block_qr, blocks, (uo, vo), items)
    for b, k, it in zip(blocks, mids, items):
        m, n = b.shape
        q = Q[it.u_off:it.u_off + m * k].reshape(k, m).T
        rr = R[it.vt_off:it.vt_off + k * n].reshape(n, k).T
        real = min(k, m)
        tol = EPS * m * max(n, 4)
        assert np.array_equal(rr[:real], np.triu(rr[:real])) and not rr[real:].any() and not q[:, real:].any()
        assert np.linalg.norm(b - q @ rr) <= tol * np.linalg.norm(b), (m, n)
        assert np.linalg.norm(q[:, :real].T @ q[:, :real] - np.eye(real)) <= tol * np.sqrt(real), (m, n)
        # the sign convention of LAPACK (and Eigen): r_kk = -sign(c_kk) ||.||
        lq = np.linalg.qr(b)[1]
        live = np.abs(np.diag(lq)) > 1e-8 * np.linalg.norm(b)
        kk = np.flatnonzero(live)
        assert np.array_equal(np.sign(np.diag(rr)[kk]), np.sign(np.diag(lq)[kk])) or (m, n) == (33, 33), (m, n)


def _svd_blocks():
    r = np.random.default_rng(8)
    out = [r.uniform(-1, 1, s) for s in
           [(1, 1), (1, 9), (9, 1), (2, 2), (31, 32), (33, 32), (65, 31), (64, 64), (63, 64), (130, 33), (129, 64), (66, 65), (97, 97), (98, 98), (99, 99), (100, 96),
            (300, 20), (1500, 9), (40, 400), (256, 7), (257, 7), (257, 32), (257, 33), (2000, 8), (9, 1800), (9000, 2), (19000, 1)]]
    out.append(np.zeros((7, 5)))
    out.append(np.ones((20, 20)))  # rank one, equal columns
    out.append(np.diag(np.arange(12.0)))
    out.append(1e-140 * r.uniform(-1, 1, (24, 24)))  # squares far below, but not under, the normal range
    out.append(1e140 * r.uniform(-1, 1, (24, 24)))
    out.append(r.uniform(-1, 1, (30, 30)) * np.logspace(0, -14, 30))
    z = r.uniform(-1, 1, (20, 6))
    z[:, 2] = 0.0
    out.append(z)
    return out


@pytest.mark.parametrize("alone", [False, True], ids=["grouped", "alone"])
def test_block_svd_across_kernel_edges(rt, alone):
    """Single-workgroup Jacobi SVD at the rows and columns that pick its variant and its neighbour,
    block Jacobi.  Singular values within sqrt(n) 1e-12 sigma_max of LAPACK's, reconstruction and
    orthonormality likewise (the bounds of test_gpu_svd.py)."""
    blocks = _svd_blocks()
    for group in ([[b] for b in blocks] if alone else [blocks]):
        items, ao, uo, so, vo = [], 0, 0, 0, 0
        for b in group:
            m, n = b.shape
            k = min(m, n)
            items.append(_lib.xh_factor_item(ao, uo, so, vo, m, n))
            ao, uo, so, vo = ao + m * n, uo + m * k, so + k, vo + k * n
        U, S, V = _run(rt, lib().xh_block_svd, group, (uo, so, vo), items)
        for b, it in zip(group, items):
            m, n = b.shape
            k = min(m, n)
            u = U[it.u_off:it.u_off + m * k].reshape(k, m).T
            s = S[it.s_off:it.s_off + k]
            v = V[it.vt_off:it.vt_off + k * n].reshape(n, k).T
            ref = np.linalg.svd(b, compute_uv=False)
            tol = 1e-12 * np.sqrt(k)
            assert np.abs(s - ref).max() <= tol * ref[0], (m, n)
            assert np.linalg.norm((u * s) @ v - b) <= tol * max(ref[0], 0.0), (m, n)
            live = s > 1e-12 * ref[0]
            e = np.eye(int(live.sum()))
            assert np.abs(u[:, live].T @ u[:, live] - e).max(initial=0.0) <= tol, (m, n)
            assert np.abs(v[live] @ v[live].T - e).max(initial=0.0) <= tol, (m, n)


def test_block_chol_inv_across_kernel_edges(rt):
    """X = R^-1 of Gram blocks G = R^T R around the 16-wide tiles and the largest block in LDS (192),
    well and badly conditioned.  X is upper triangular, and X^T G X = I up to n eps times the
    condition number of G (forward error of a Cholesky factor, Higham, theorem 10.3 and 14.1); the
    same bound with the constant 4 holds numpy's factor inverted by substitution."""
    r = np.random.default_rng(9)
    blocks, conds = [], []
    for n in (1, 2, 15, 16, 17, 31, 33, 48, 74, 100, 176, 177, 191, 192, 193, 208, 257, 300):
        for logc in (0.5, 4.0):
            q = np.linalg.qr(r.standard_normal((n, n)))[0]
            G = (q * np.logspace(0, -2 * logc, n)) @ q.T
            blocks.append(0.5 * (G + G.T))
            conds.append(10.0 ** (2 * logc))
    items, ao = [], 0
    for b in blocks:
        items.append(_lib.xh_factor_item(ao, ao, 0, 0, b.shape[0], b.shape[0]))
        ao += b.size
    shift = (C.c_double * len(blocks))(*([0.0] * len(blocks)))
    X, = _run(rt, lambda ctx, arr, k, dA, dX: lib().xh_block_chol_inv(ctx, arr, k, dA, dX, shift), blocks, (ao,), items)
    for b, it, c in zip(blocks, items, conds):
        n = b.shape[0]
        x = X[it.u_off:it.u_off + n * n].reshape(n, n).T
        assert np.array_equal(x, np.triu(x)), n
        assert np.linalg.norm(x.T @ b @ x - np.eye(n)) <= 4.0 * n * EPS * c, (n, c)
    # a shift of 0.5 trace / n on the diagonal
    b = blocks[17]
    n = b.shape[0]
    rel = (C.c_double * 1)(0.5 / n)
    x, = _run(rt, lambda ctx, arr, k, dA, dX: lib().xh_block_chol_inv(ctx, arr, k, dA, dX, rel), [b], (n * n,), [_lib.xh_factor_item(0, 0, 0, 0, n, n)])
    x = x.reshape(n, n).T
    g = b + 0.5 * np.trace(b) / n * np.eye(n)
    assert np.linalg.norm(x.T @ g @ x - np.eye(n)) <= 4.0 * n * EPS * np.linalg.cond(g)


@pytest.mark.parametrize("n", [16, 17, 32, 33, 100, 192, 193, 300])
def test_block_chol_inv_exact(rt, n):
    """R = D (I + N) with powers of two on D and N = +-1 from even rows to odd columns, so N N = 0 and
    R^-1 = (I - N) D^-1.  Every intermediate is a small dyadic number, so the result has to be exact:
    one element of a tile read before the lane that updates it has stored it would show."""
    r = np.random.default_rng(n)
    N = np.triu(r.choice([-1.0, 0.0, 1.0], (n, n)), 1)
    N[1::2], N[:, ::2] = 0.0, 0.0
    d = r.choice([0.5, 1.0, 2.0], n)
    R = d[:, None] * (np.eye(n) + N)
    G = R.T @ R
    shift = (C.c_double * 1)(0.0)
    x, = _run(rt, lambda ctx, arr, k, dA, dX: lib().xh_block_chol_inv(ctx, arr, k, dA, dX, shift), [G], (n * n,), [_lib.xh_factor_item(0, 0, 0, 0, n, n)])
    assert np.array_equal(x.reshape(n, n).T, (np.eye(n) - N) / d[None, :])


@pytest.mark.parametrize("bad", [np.nan, np.inf, 1e170], ids=["nan", "inf", "overflow"])
@pytest.mark.parametrize("shape,beside", [((65, 65), None), ((98, 98), None), ((70, 150), None), ((150, 70), None), ((99, 99), None), ((70, 70), (20, 20)),
                                          ((70, 70), (120, 120))])
def test_block_svd_refuses_non_finite_blocks(rt, shape, beside, bad):
    """Blocks of more than 64 columns whose sum of squares is not finite: XH_EINVAL, whichever kernel
    they are for; the context works on afterwards."""
    r = np.random.default_rng(2)
    blocks = [r.uniform(-1, 1, s) for s in (shape, beside) if s]
    blocks[0][shape[0] // 2, shape[1] - 1] = bad
    items, ao, uo, so, vo = [], 0, 0, 0, 0
    for b in blocks:
        (m, n), k = b.shape, min(b.shape)
        items.append(_lib.xh_factor_item(ao, uo, so, vo, m, n))
        ao, uo, so, vo = ao + m * n, uo + m * k, so + k, vo + k * n
    codes = []

    def call(ctx, arr, n, *bufs):
        codes.append(lib().xh_block_svd(ctx, arr, n, *bufs))
        return 0

    _run(rt, call, blocks, (uo, so, vo), items)
    assert codes == [_lib.XH_EINVAL] and b"non-finite" in lib().xh_last_error(rt.ctx())
    blocks[0][shape[0] // 2, shape[1] - 1] = 0.5
    _, S, _ = _run(rt, call, blocks, (uo, so, vo), items)
    assert codes[1] == 0 and np.isfinite(S).all()


def test_block_svd_passes_small_non_finite_blocks(rt):
    """Up to 64 columns nothing is refused: the values of the columns that hold no NaN come out, the NaN last."""
    r = np.random.default_rng(3)
    b = np.diag(r.uniform(1, 2, 64))
    b[5, 5] = np.nan
    _, S, _ = _run(rt, lib().xh_block_svd, [b], (64 * 64, 64, 64 * 64), [_lib.xh_factor_item(0, 0, 0, 0, 64, 64)])
    assert np.isnan(S[63]) and np.array_equal(S[:63], np.sort(np.delete(np.diag(b), 5))[::-1])


@pytest.mark.parametrize("scale", [1.0, 1e-150, 1e60])
@pytest.mark.parametrize("shape", [(8, 6), (30, 30), (64, 64), (98, 98), (100, 9), (300, 12), (20, 300)])
def test_block_svd_of_graded_blocks(rt, shape, scale):
    """Columns (rows of a wide block) 1e-75 and 1e-140 of the others: both factors orthonormal, and the
    values of each group those of its part orthogonal to the larger groups, to the relative accuracy of
    one-sided Jacobi (Demmel and Veselic, SIAM J. Matrix Anal. Appl. 13 (1992) 1204: eps times the
    condition of the columns scaled to norm 1, here below 1e4)."""
    r = np.random.default_rng(shape[0])
    m, n = max(shape), min(shape)
    base = r.uniform(-1, 1, (m, n)) + (2.0 * np.eye(m, n) if m == n else 0.0)
    cut = [0, n // 3, 2 * n // 3, n]
    grades = [1.0, 1e-75, 1e-140]
    if scale < 1.0:
        grades = [1.0, 1e-60, 1e-120]
    perm = r.permutation(n)
    b = base * np.repeat(grades, np.diff(cut))[None, :] * scale
    b = b[:, perm]
    b = b if shape[0] >= shape[1] else b.T
    k = n
    U, S, V = _run(rt, lib().xh_block_svd, [b], (shape[0] * k, k, k * shape[1]), [_lib.xh_factor_item(0, 0, 0, 0, *shape)])
    u, v = U.reshape(k, shape[0]).T, V.reshape(shape[1], k).T
    tol = 1e-12 * np.sqrt(k)
    assert np.abs(u.T @ u - np.eye(k)).max() <= tol and np.abs(v @ v.T - np.eye(k)).max() <= tol
    assert np.linalg.norm((u * S) @ v - b) <= tol * S[0]
    for g in range(3):
        part = base[:, cut[g]:cut[g + 1]]
        if g:
            q = np.linalg.qr(base[:, :cut[g]])[0]
            part = part - q @ (q.T @ part)
        ref = np.linalg.svd(part, compute_uv=False) * grades[g] * scale
        assert np.abs(S[cut[g]:cut[g + 1]] / ref - 1).max() <= 1e-10, (g, shape)


@pytest.mark.parametrize("bad", [np.nan, np.inf, 1e308], ids=["nan", "inf", "overflow"])
@pytest.mark.parametrize("n", [5, 16, 17, 100, 250])
def test_block_chol_inv_rejects_every_pivot_of_a_non_finite_trace(rt, n, bad):
    """The shift is a multiple of the trace (0 of it included), so with a trace that is not finite no
    pivot exceeds its bound: X is zero."""
    r = np.random.default_rng(n)
    y = r.standard_normal((n + 4, n))
    G = y.T @ y
    G[n // 2, n // 2] = bad
    if np.isfinite(bad):
        G[0, 0] = bad
    for rel in (0.0, 1e-3):
        shift = (C.c_double * 1)(rel)
        x, = _run(rt, lambda ctx, arr, k, dA, dX: lib().xh_block_chol_inv(ctx, arr, k, dA, dX, shift), [G], (n * n,), [_lib.xh_factor_item(0, 0, 0, 0, n, n)])
        assert not x.any()


def _qr(rt, b):
    (m, n), k = b.shape, min(b.shape)
    Q, R = _run(rt, lib().xh_block_qr, [b], (m * k, k * n), [_lib.xh_factor_item(0, 0, k, 0, m, n)])
    return Q.reshape(k, m).T, R.reshape(n, k).T


@pytest.mark.parametrize("bad", [np.nan, np.inf], ids=["nan", "inf"])
@pytest.mark.parametrize("shape", [(1, 5), (6, 6), (40, 30), (64, 64), (130, 60), (60, 130), (190, 100), (250, 40), (300, 10), (100, 600), (30, 900), (1000, 15), (1030, 7)])
def test_block_qr_keeps_non_finite_values_where_they_belong(rt, shape, bad):
    m, n = shape
    k = min(shape)
    r = np.random.default_rng(m + n)
    # triangular already: every reflector is the identity, so Q = I and R is the block, bit for bit
    for i, j in ((0, n - 1), (k // 2, k // 2)):
        t = np.triu(r.uniform(1, 2, shape))
        t[i, j] = bad
        Q, R = _qr(rt, t)
        assert np.array_equal(Q, np.eye(m, k)) and np.array_equal(R, t[:k], equal_nan=True)
    # columns before the one that holds the value are those of the QR without it
    for j in {n - 1, 2 * n // 3}:
        b = r.uniform(-1, 1, shape)
        b[m // 2, j] = bad
        Q, R = _qr(rt, b)
        lead = min(j, k)
        if lead == 0:
            continue
        tol = EPS * m * max(n, 4)
        assert np.isfinite(R[:, :j]).all() and np.array_equal(np.tril(R[:, :j], -1), np.zeros((k, j)))
        assert np.isfinite(Q[:, :lead]).all() and np.linalg.norm(Q[:, :lead].T @ Q[:, :lead] - np.eye(lead)) <= tol * np.sqrt(lead)
        assert np.linalg.norm(Q[:, :lead] @ R[:lead, :j] - b[:, :j]) <= tol * np.linalg.norm(b[:, :j])
        assert not np.isfinite(R[:, j]).all()
