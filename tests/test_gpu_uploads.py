"""Item lists of a call around the sizes at which their way to the device changes (504 bytes, and lengths
that are no multiple of 8), exact results (needs an MI355X)."""
import ctypes as C

import numpy as np
import pytest

from xped_amd._lib import lib

pytestmark = pytest.mark.gpu


def _on_device(rt, x):
    p = C.c_void_p()
    assert lib().xh_alloc(rt.ctx(), x.nbytes, C.byref(p)) == 0
    lib().xh_upload(rt.ctx(), p, x.ctypes.data, x.nbytes)
    return p


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 63, 64, 65, 287, 288, 289, 321, 1001])
def test_offsets_and_sizes(rt, n):
    """Two lists in one upload, 8 n bytes and 4 n bytes from the next multiple of 256 on."""
    L, ctx = lib(), rt.ctx()
    m = (np.arange(n) % 3 + 1).astype(np.int32)
    off = np.concatenate([[0], np.cumsum(m.astype(np.int64) ** 2)])
    x = 2.0 ** (np.arange(off[-1]) % 7)
    p = _on_device(rt, x)
    diag_map = L.xh_block_diag_map
    diag_map.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_int64, C.c_void_p, C.c_int]
    assert diag_map(ctx, off.ctypes.data, m.ctypes.data, n, p, 1) == 0
    out = np.empty_like(x)
    L.xh_download(ctx, out.ctypes.data, p, x.nbytes)
    L.xh_free(ctx, p)
    for o, k in zip(off, m):
        x[o:o + k * k:k + 1] = 1.0 / x[o:o + k * k:k + 1]
    assert np.array_equal(out, x)


@pytest.mark.parametrize("n", [1, 31, 32, 33, 223, 224, 225])
def test_ranges(rt, n):
    L, ctx = lib(), rt.ctx()
    ln = np.arange(n, dtype=np.int64) % 5
    off = np.concatenate([[0], np.cumsum(ln)])[:-1].copy()
    x = np.arange(int(ln.sum()) + 1, dtype=float)
    p = _on_device(rt, x)
    out = np.empty(n)
    i64 = C.POINTER(C.c_int64)
    assert L.xh_range_sumsq(ctx, off.ctypes.data_as(i64), ln.ctypes.data_as(i64), n, p, out.ctypes.data_as(C.POINTER(C.c_double))) == 0
    L.xh_free(ctx, p)
    assert np.array_equal(out, [np.sum(x[o:o + k] ** 2) for o, k in zip(off, ln)])


@pytest.mark.parametrize("transpose", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 70])
def test_rectangles(rt, n, transpose):
    """Up to 16 rectangles are kernel arguments, more are uploaded."""
    L, ctx = lib(), rt.ctx()
    r = np.random.default_rng(n)

    class Rect(C.Structure):
        _fields_ = [("src_off", C.c_int64), ("src_ld", C.c_int64), ("dst_off", C.c_int64), ("dst_ld", C.c_int64), ("rows", C.c_int32), ("cols", C.c_int32),
                    ("factor", C.c_double), ("transpose", C.c_int32)]

    src, rects, at = r.uniform(-1, 1, 5000), [], 0
    for q in range(n):
        m, k = int(r.integers(0, 40)), int(r.integers(1, 40))
        rects.append(Rect(int(r.integers(0, 1000)), (k if transpose else m) + q % 3, at, m + q % 2, m, k, 1.0 if q % 2 else -2.0, transpose))
        at += (m + q % 2) * k
    out = np.full(max(at, 1), 7.0)
    exp, a, b = out.copy(), _on_device(rt, src), _on_device(rt, out)
    copy = L.xh_copy_rects
    copy.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_int64]
    assert copy(ctx, a, b, C.addressof((Rect * n)(*rects)), n) == 0
    L.xh_download(ctx, out.ctypes.data, b, out.nbytes)
    L.xh_free(ctx, a)
    L.xh_free(ctx, b)
    for x in rects:
        i, j = np.meshgrid(np.arange(x.rows), np.arange(x.cols), indexing="ij")
        exp[x.dst_off + i + j * x.dst_ld] = x.factor * src[x.src_off + (j + i * x.src_ld if transpose else i + j * x.src_ld)]
    assert np.array_equal(out, exp)
