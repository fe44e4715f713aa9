"""Item lists of a call around the sizes at which their way to the device changes (512 and 3584 bytes,
and lengths that are no multiple of 8), exact results (needs an MI355X)."""
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
