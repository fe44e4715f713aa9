"""FP64 grouped GEMM at the edges of its tile shapes (needs an MI355X): output sides around 32, 64,
96, 128 and 192, K around the steps of 8 and 16 and with a split K, all four transposes, against
numpy.  Bound: |error| <= k u |A| |B| elementwise (Higham, Accuracy and Stability of Numerical
Algorithms, 2nd ed., section 3.5), doubled for the reference's own.  Non-finite entries reach only
the rows and columns that hold them: tiles read past a matrix's last row and the end of K, into
neighbouring values."""
import ctypes as C

import numpy as np
import pytest
import torch

from xped_amd import _lib
from xped_amd._lib import lib

pytestmark = pytest.mark.gpu

U = 2.0 ** -53
SIDES = [1, 31, 32, 33, 64, 65, 95, 96, 97, 128, 129, 191, 193, 200, 257]


def _workspace(rt, shapes, ta=0, tb=0):
    """Device bytes of the split-K partials of a plan."""
    L, plan, b = lib(), C.c_void_p(), C.c_int64()
    items = (_lib.xh_gemm_item * len(shapes))(*[_lib.xh_gemm_item(0, 0, 0, *s) for s in shapes])
    assert L.xh_gemm_plan_create(rt.ctx(), items, len(shapes), ta, tb, C.byref(plan)) == 0
    assert L.xh_gemm_plan_workspace(plan, C.byref(b)) == 0
    L.xh_gemm_plan_destroy(rt.ctx(), plan)
    return b.value


def _products(rt, mats, ta, tb, gemm=None):
    """C of every (A, B) in one grouped call; operands stored column-major, transposed where asked."""
    L, ctx = lib(), rt.ctx()
    items, ao, bo, co, fa, fb = [], 0, 0, 0, [], []
    for A, B in mats:
        m, k = A.shape
        n = B.shape[1]
        items.append(_lib.xh_gemm_item(ao, bo, co, m, n, k))
        fa.append((A if ta else A.T).reshape(-1))
        fb.append((B if tb else B.T).reshape(-1))
        ao, bo, co = ao + m * k, bo + k * n, co + m * n
    bufs = [C.c_void_p() for _ in range(3)]
    for p, n in zip(bufs, (ao, bo, co)):
        assert L.xh_alloc(ctx, 8 * n, C.byref(p)) == 0
    for p, x in ((bufs[0], np.concatenate(fa)), (bufs[1], np.concatenate(fb))):
        x = np.ascontiguousarray(x)
        L.xh_upload(ctx, p, x.ctypes.data, 8 * x.size)
    arr = (_lib.xh_gemm_item * len(items))(*items)
    plan = C.c_void_p()
    assert L.xh_gemm_plan_create(ctx, arr, len(items), ta, tb, C.byref(plan)) == 0
    assert (gemm or L.xh_gemm)(ctx, plan, *bufs, 1.0, 0.0, _lib.XH_FP64) == 0, L.xh_last_error(ctx)
    out = np.empty(co)
    L.xh_download(ctx, out.ctypes.data, bufs[2], 8 * co)
    L.xh_gemm_plan_destroy(ctx, plan)
    for p in bufs:
        L.xh_free(ctx, p)
    return [out[it.c_off:it.c_off + it.m * it.n].reshape(it.n, it.m).T for it in items]


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("ks", [(33, 48, 64, 200), (35, 47, 63, 129), (777,)], ids=["even", "odd", "split"])
def test_tile_shapes(rt, ta, tb, ks):
    r = np.random.default_rng(3)
    sides = SIDES if len(ks) > 1 else SIDES[:7]
    shapes = [(m, n, ks[(i + j) % len(ks)]) for i, m in enumerate(sides) for j, n in enumerate(sides)]
    mats = [(r.uniform(-1, 1, (m, k)), r.uniform(-1, 1, (k, n))) for m, n, k in shapes]
    for (A, B), c in zip(mats, _products(rt, mats, ta, tb)):
        assert np.all(np.abs(c - A @ B) <= 2 * A.shape[1] * U * (np.abs(A) @ np.abs(B))), (A.shape, B.shape)


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_nonfinite_entries_stay_in_their_rows_and_columns(rt, ta, tb):
    r = np.random.default_rng(4)
    mats, clean = [], []
    for m, n, k in [(65, 70, 41), (97, 33, 43), (193, 257, 35), (70, 300, 47), (40, 40, 519)]:
        A, B = r.uniform(-1, 1, (m, k)), r.uniform(-1, 1, (k, n))
        A[5, :3], A[m - 1, 0], B[:2, 7], B[0, n - 1] = np.nan, np.inf, np.nan, -np.inf
        mats.append((A, B))
        rows, cols = np.ones(m, bool), np.ones(n, bool)
        rows[[5, m - 1]] = cols[[7, n - 1]] = False
        clean.append((rows, cols))
    for (A, B), (rows, cols), c in zip(mats, clean, _products(rt, mats, ta, tb)):
        ref = A[rows] @ B[:, cols]
        assert np.all(np.abs(c[np.ix_(rows, cols)] - ref) <= 2 * A.shape[1] * U * (np.abs(A[rows]) @ np.abs(B[:, cols])))
        assert not np.isfinite(c[~rows]).any() and not np.isfinite(c[:, ~cols]).any()


def test_operands_beyond_32_bit_tile_offsets(rt):
    # K of 2.1 million: 128 rows of a K-contiguous operand span more than 2 GiB, so the item takes
    # the tiles with checked 64-bit loads (three rows keep the operands small)
    r = np.random.default_rng(5)
    k = 2_100_000
    A, B = r.uniform(-1, 1, (3, k)), r.uniform(-1, 1, (k, 2))
    c, = _products(rt, [(A, B)], 1, 0)
    assert np.all(np.abs(c - A @ B) <= 2 * k * U * (np.abs(A) @ np.abs(B)))


@pytest.mark.parametrize("shape", [(74, 74, 3000), (500, 500, 500)])
def test_short_items_do_not_take_the_k_split_from_long_ones(rt, shape):
    """The partial products of a call (its split along K) are those of its long items alone, however many
    items of 256 x 16 x 16 run as tiles beside them."""
    alone = _workspace(rt, [shape])
    assert alone > 0 and [_workspace(rt, [shape] + [(256, 16, 16)] * s) for s in (1, 100, 400, 2000)] == [alone] * 4


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 1)])
def test_split_has_no_more_chunks_than_plain_tiles_give(rt, ta, tb):
    """Partials of a plan, whatever its tile shapes, against the split that 64 x 64 tiles (128 x 128 from 192
    a side) give: chunks for 4 tiles per CU, of at least 128 in multiples of 16."""
    target = 4 * torch.cuda.get_device_properties(0).multi_processor_count

    def bound(shapes):
        tiles = sum(-(-m // t) * -(-n // t) for m, n, _ in shapes for t in [128 if min(m, n) >= 192 else 64])
        chunks = -(-target // tiles) if tiles < target else 1
        total = 0
        for m, n, k in shapes:
            kc = max(128, (-(-k // chunks) + 15) // 16 * 16)
            if chunks > 1 and k >= 256 and -(-k // kc) > 1:
                total += 8 * m * n * -(-k // kc)
        return total

    sides = [33, 65, 74, 96, 97, 130, 192, 200, 260, 390, 700, 1900]
    for m in sides:
        for n in sides:
            for k in (300, 2000, 8000):
                for count in (1, 5, 18):
                    assert _workspace(rt, [(m, n, k)] * count, ta, tb) <= bound([(m, n, k)] * count), (m, n, k, count)
    assert _workspace(rt, [(1900, 74, 500)] * 18, ta, tb) == 0  # not split, so it may be captured


def test_noalloc_takes_a_long_sketch_product(rt):
    """1900 x 74 with K = 8000 has partials below the array's 32 MiB."""
    r = np.random.default_rng(4)
    A, B = r.uniform(-1, 1, (1900, 8000)), r.uniform(-1, 1, (8000, 74))
    c, = _products(rt, [(A, B)], 0, 0, lib().xh_gemm_noalloc)
    assert np.all(np.abs(c - A @ B) <= 2 * A.shape[1] * U * (np.abs(A) @ np.abs(B)))
