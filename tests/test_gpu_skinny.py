"""Skinny FP64 products (short side and K at most 32) and the gather product at their edges (needs an
MI355X), against numpy within k u |A| |B| elementwise (Higham, Accuracy and Stability of Numerical
Algorithms, 2nd ed., section 3.5), doubled for the reference's own: K around the multiples of 4,
short sides around the sums of one pass, calls whose short sides are all at most 8 (scalar operands)
and others (operands from LDS), all transposes, non-finite entries, domain legs that drop out, join
and do not, several domain trees per workgroup, source strides past 32 bits."""
import ctypes as C

import numpy as np
import pytest

from xped_amd import _lib
from xped_amd._lib import lib

from .test_gpu_gemm_tiles import U, _products

pytestmark = pytest.mark.gpu

SHORT = [1, 2, 3, 4, 5, 8, 9, 17, 31, 32]


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("short", [SHORT, [1, 2, 3, 4, 5, 7, 8]], ids=["s32", "s8"])
@pytest.mark.parametrize("ks", [(1, 3, 4, 5, 8, 9, 11, 12, 13, 16), (17, 20, 21, 24, 25, 28, 29, 31, 32)], ids=["k16", "k32"])
def test_skinny_products(rt, ta, tb, ks, short):
    r = np.random.default_rng(5)
    mats = []
    for i, k in enumerate(ks):
        for j, s in enumerate(short):
            long = (33, 256, 257, 700)[(i + j) % 4]
            m, n = (s, long) if (i + j // 2) % 2 else (long, s)
            A, B = r.uniform(-1, 1, (m, k)), r.uniform(-1, 1, (k, n))
            if j % 3 == 0:  # in the last term: what follows it in memory is a neighbour's
                A[m // 2, k - 1], B[0, n - 1] = np.inf, np.nan
            mats.append((A, B))
    for (A, B), c in zip(mats, _products(rt, mats, ta, tb)):
        rows, cols = np.isfinite(A).all(axis=1), np.isfinite(B).all(axis=0)
        A1, B1 = A[rows], B[:, cols]
        assert np.all(np.abs(c[np.ix_(rows, cols)] - A1 @ B1) <= 2 * A.shape[1] * U * (np.abs(A1) @ np.abs(B1))), (A.shape, B.shape)
        assert not np.isfinite(c[~rows]).any() and not np.isfinite(c[:, ~cols]).any()


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("k", [7, 16, 23, 32])
def test_skinny_variants_same_bits(rt, ta, tb, k):
    """The variant follows the largest short side and K of the call; an item's sums do not."""
    r = np.random.default_rng(k)
    mats = [(r.uniform(-1, 1, (m, k)), r.uniform(-1, 1, (k, n))) for m, n in ((500, 8), (3, 300), (700, 1), (6, 257))]
    wide = [(r.uniform(-1, 1, (400, kw)), r.uniform(-1, 1, (kw, 32))) for kw in (k, 32)]
    alone = _products(rt, mats, ta, tb)
    for w in wide:
        for a, b in zip(alone, _products(rt, mats + [w], ta, tb)):
            assert np.array_equal(a, b)


class _GatherItem(C.Structure):
    _fields_ = [("task_base", C.c_int32), ("ndom", C.c_int32), ("ncod", C.c_int32), ("pad", C.c_int32), ("starts_off", C.c_int64)]


class _GatherDesc(C.Structure):
    _fields_ = [("perm", _lib.xh_permute_desc), ("nitems", C.c_int64), ("items", C.POINTER(_GatherItem)), ("nstarts", C.c_int64),
                ("starts", C.POINTER(C.c_int32)), ("src_elems", C.c_int64)]


@pytest.mark.parametrize("far", [0, 1 << 32], ids=["near", "far"])
@pytest.mark.parametrize("ns", [(1, 3, 8, 11), (1, 5, 8), (17, 32)], ids=["n11", "n8", "n32"])
@pytest.mark.parametrize("kmax", [12, 32])
def test_gather_product(rt, kmax, ns, far):
    gather_product(rt, kmax, ns, far, 40)


def test_gather_product_of_many_trees(rt):
    """Plan tables filled by several host threads."""
    gather_product(rt, 16, (3,), 0, 8000)


def gather_product(rt, kmax, ns, far, ntrees):
    """far: one domain leg of extent 2 whose source entries lie 2^32 elements apart (a 34 GB source)."""
    r = np.random.default_rng(kmax)
    L, ctx = lib(), rt.ctx()
    NL, NR, W = 5, 3, 1 << 20
    src = r.uniform(-1, 1, W)
    tasks, sources, starts, gitems, gemms, ops = [], [], [], [], [], []
    bo = co = 0
    for n in ns:
        dom = [[int(x) for x in (r.choice([1, 2, 45]), r.choice([1, 3]), 2 if far else r.choice([1, 2, 7]))] for _ in range(ntrees)]
        cod = []
        while sum(a * b for a, b in cod) < kmax - 4:
            cod.append((int(r.integers(1, 3)), int(r.integers(1, 3))))
        ds, cs = np.cumsum([0] + [int(np.prod(x)) for x in dom]), np.cumsum([0] + [a * b for a, b in cod])
        m, k = int(ds[-1]), int(cs[-1])
        gitems.append(_GatherItem(len(tasks), len(dom), len(cod), 0, len(starts)))
        starts += [int(x) for x in ds] + [int(x) for x in cs]
        A = np.empty((m, k))
        for a, de in enumerate(dom):
            for b, ce in enumerate(cod):
                e = de + list(ce)
                if far:  # domain legs 0 and 1 joined, leg 2 along the source's columns
                    st, col, ld = [1, e[0], 1, e[0] * e[1], e[0] * e[1] * e[3]], [0, 0, 1, 0, 0], far
                else:
                    order = [int(x) for x in ((0, 1, 2, 3, 4) if a % 2 else r.permutation(5))]
                    st, col, mult, cut = [0] * 5, [0] * 5, [1, 1], int(r.integers(1, 5))
                    for i, q in enumerate(order):
                        st[q], col[q] = mult[i >= cut], int(i >= cut)
                        mult[i >= cut] *= e[q]
                    ld = mult[0] + int(r.integers(0, 3))
                off, coeff = int(r.integers(0, W // 2)), float(r.choice([1.0, -1.0]))
                tasks.append(_lib.xh_permute_task(0, e[0] * e[1] * e[2], e[0] * e[1] * e[2], e[3] * e[4], 1, len(sources), (C.c_uint32 * _lib.XH_MAXLEGS)(*e),
                                                  (C.c_int64 * _lib.XH_MAXLEGS)(*st), (C.c_uint8 * _lib.XH_MAXLEGS)(*col)))
                sources.append(_lib.xh_permute_source(off, ld, coeff))
                at = np.full(1, off)
                for q in range(5):  # the far column is the near one shifted by 7
                    step = st[q] * ((7 if far else ld) if col[q] else 1)
                    at = (at[None, :] + step * np.arange(e[q])[:, None]).reshape(-1)
                A[ds[a]:ds[a + 1], cs[b]:cs[b + 1]] = coeff * src[at].reshape(e[3] * e[4], -1).T
        gemms.append(_lib.xh_gemm_item(0, bo, co, m, n, k))
        ops.append((A, r.uniform(-1, 1, (k, n))))
        bo, co = bo + k * n, co + m * n
    n_src = far + W if far else W
    arrays = [(_lib.xh_permute_task * len(tasks))(*tasks), (_lib.xh_permute_source * len(sources))(*sources), (_GatherItem * len(gitems))(*gitems),
              (C.c_int32 * len(starts))(*starts), (_lib.xh_gemm_item * len(gemms))(*gemms)]
    gemm, plan, bufs = C.c_void_p(), C.c_void_p(), [C.c_void_p() for _ in range(3)]
    assert L.xh_gemm_plan_create(ctx, arrays[4], len(gemms), 0, 0, C.byref(gemm)) == 0
    desc = _GatherDesc(_lib.xh_permute_desc(NL, NR, len(tasks), len(sources), arrays[0], arrays[1]), len(gitems), arrays[2], len(starts), arrays[3], n_src)
    assert L.xh_gather_plan_create(ctx, gemm, C.byref(desc), C.byref(plan)) == 0, L.xh_last_error(ctx)
    for p, n in zip(bufs, (n_src, bo, co)):
        assert L.xh_alloc(ctx, 8 * n, C.byref(p)) == 0
    L.xh_upload(ctx, bufs[0], src.ctypes.data, src.nbytes)
    if far:
        shifted = np.roll(src, -7)
        L.xh_upload(ctx, C.c_void_p(bufs[0].value + 8 * far), shifted.ctypes.data, src.nbytes)
    B = np.concatenate([b.T.reshape(-1) for _, b in ops])
    L.xh_upload(ctx, bufs[1], B.ctypes.data, B.nbytes)
    out = np.empty(co)
    assert L.xh_gemm_gather(ctx, gemm, plan, bufs[0], n_src, bufs[1], bufs[2], 1.0, 0.0) == 0, L.xh_last_error(ctx)
    L.xh_download(ctx, out.ctypes.data, bufs[2], out.nbytes)
    L.xh_gather_plan_destroy(ctx, plan)
    L.xh_gemm_plan_destroy(ctx, gemm)
    for p in bufs:
        L.xh_free(ctx, p)
    for it, (a, b) in zip(gemms, ops):
        c = out[it.c_off:it.c_off + it.m * it.n].reshape(it.n, it.m).T
        assert np.all(np.abs(c - a @ b) <= 2 * it.k * U * (np.abs(a) @ np.abs(b)))
