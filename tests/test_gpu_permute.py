"""The grouped permute from descriptors against numpy (needs an MI355X): bit for bit where an element
has one source with a coefficient +-1, and within n u sum |c v| (u = 2^-53, n sources; a product may
be fused with its sum on one side alone, hence twice that) where it sums several.  Both gathers
(compact tasks, and the general one for source indices of 2^31 and more) and the transpose tasks
beside them.  Legs of extent 1, legs that join and legs that do not, more legs than a workgroup
stages, one element to thousands of tasks per workgroup, source lists in any order, both tile sizes."""
import ctypes as C

import numpy as np
import pytest

from xped_amd import _lib
from xped_amd._lib import lib

pytestmark = pytest.mark.gpu


def _task(r, nlegs, new_rank, exts, nsrc, p_join):
    """Output leg extents, their source strides (a random order of the source's row and column legs)
    and the source's shape."""
    e = [int(r.choice(exts)) for _ in range(nlegs)]
    order = list(range(nlegs)) if r.random() < p_join else [int(x) for x in r.permutation(nlegs)]
    cut = new_rank if r.random() < 0.5 else int(r.integers(0, nlegs + 1))
    st, col = [0] * nlegs, [0] * nlegs
    rows = cols = 1
    for i, q in enumerate(order):
        if i < cut:
            st[q], rows = rows, rows * e[q]
        else:
            st[q], col[q], cols = cols, 1, cols * e[q]
    return e, st, col, rows, cols, nsrc


def _run(rt, tasks, nlegs, new_rank, shuffled=False, far=0):
    """Runs the tasks on one source buffer and compares with numpy.  far > 0: each source's leading dimension."""
    r = np.random.default_rng(len(tasks))
    L, ctx = lib(), rt.ctx()
    src, recs, sources, so_of, dst_off = r.uniform(-1, 1, 1 << 16), [], [], [], 3
    src[::97] = 0.0
    src[5::97] = -0.0
    expected = {}
    blocks = [[] for _ in tasks]
    for i in (r.permutation(len(tasks)) if shuffled else range(len(tasks))):
        e, st, col, rows, cols, nsrc = tasks[i]
        begin = len(sources)
        for _ in range(nsrc):
            ld = far or rows + int(r.integers(0, 3))
            off = int(r.integers(0, 1 << 15))
            sources.append((off, ld, float(r.choice([1.0, -1.0] if nsrc == 1 else [0.37, -1.25, 0.5]))))
        blocks[i] = (begin, nsrc)
    need = 1 << 16
    if not far:
        need = 1 + max([(1 << 15) + (t[3] + 2) * t[4] for t in tasks])
        src = np.resize(src, max(need, src.size))
    want = []
    for i, (e, st, col, rows, cols, nsrc) in enumerate(tasks):
        m, n = int(np.prod(e[:new_rank], dtype=np.int64)), int(np.prod(e[new_rank:], dtype=np.int64))
        ld = m + i % 2
        recs.append(_lib.xh_permute_task(dst_off, ld, m, n, nsrc, blocks[i][0], (C.c_uint32 * _lib.XH_MAXLEGS)(*e),
                                         (C.c_int64 * _lib.XH_MAXLEGS)(*st), (C.c_uint8 * _lib.XH_MAXLEGS)(*col)))
        row, colx = np.zeros(1, np.int64), np.zeros(1, np.int64)
        for q in range(nlegs):  # column-major over the output legs
            j = np.arange(e[q])
            row = (row[None, :] + (0 if col[q] else st[q]) * j[:, None]).reshape(-1)
            colx = (colx[None, :] + (st[q] if col[q] else 0) * j[:, None]).reshape(-1)
        acc, mag = np.zeros(m * n), np.zeros(m * n)
        for s in range(blocks[i][0], blocks[i][0] + nsrc):
            o, sld, c = sources[s]
            v = src[(o + row + 7 * colx) % (1 << 16)] if far else src[o + row + colx * sld]
            acc, mag = acc + c * v, mag + np.abs(c * v)
        want.append((dst_off, ld, m, n, acc, 2 * nsrc * 2.0 ** -53 * mag if nsrc > 1 else 0.0 * mag))
        dst_off += ld * n + i % 3
    S = (_lib.xh_permute_source * max(len(sources), 1))(*[_lib.xh_permute_source(*s) for s in sources])
    T = (_lib.xh_permute_task * len(recs))(*recs)
    plan, a, b = C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert L.xh_permute_plan_create(ctx, C.byref(_lib.xh_permute_desc(nlegs, new_rank, len(recs), len(sources), T, S)), C.byref(plan)) == 0
    n_src = src.size if not far else far + (1 << 16)
    assert L.xh_alloc(ctx, 8 * n_src, C.byref(a)) == 0 and L.xh_alloc(ctx, 8 * dst_off, C.byref(b)) == 0
    L.xh_upload(ctx, a, src.ctypes.data, 8 * src.size)
    if far:  # column 1 lies far elements on: the first one shifted by 7
        shifted = np.roll(src, -7)
        L.xh_upload(ctx, C.c_void_p(a.value + 8 * far), shifted.ctypes.data, 8 * src.size)
    out = np.full(dst_off, 99.0)
    exp = out.copy()
    L.xh_upload(ctx, b, out.ctypes.data, out.nbytes)
    assert L.xh_permute(ctx, plan, a, b) == 0, L.xh_last_error(ctx)
    L.xh_download(ctx, out.ctypes.data, b, out.nbytes)
    L.xh_permute_plan_destroy(ctx, plan)
    L.xh_free(ctx, a)
    L.xh_free(ctx, b)
    tol = np.zeros(dst_off)
    for off, ld, m, n, acc, bound in want:
        for j in range(n):
            exp[off + j * ld:off + j * ld + m] = acc[j * m:(j + 1) * m]
            tol[off + j * ld:off + j * ld + m] = bound[j * m:(j + 1) * m]
    assert np.all(np.abs(out - exp) <= tol)
    assert np.array_equal(out[tol == 0].view(np.int64), exp[tol == 0].view(np.int64))


@pytest.mark.parametrize("nsrc", [(1,), (1, 2, 3, 9), (0, 1)], ids=["single", "several", "empty"])
@pytest.mark.parametrize("nlegs,new_rank,exts,ntasks", [
    (0, 0, [1], 3), (1, 1, [1, 5], 700), (4, 2, [1], 1030), (4, 2, [1, 2], 900), (4, 2, [1, 3, 17], 60), (5, 0, [1, 4], 47), (5, 5, [2, 3], 49),
    (7, 3, [1, 2, 5], 200), (20, 9, [1, 1, 2], 40), (12, 5, [2], 5), (3, 1, [40, 70], 30), (3, 2, [90, 110], 2),
    (10, 4, [3], 2), (9, 3, [2, 4], 3), (2, 1, [1, 2, 3], 17000)])
def test_against_numpy(rt, nlegs, new_rank, exts, ntasks, nsrc):
    r = np.random.default_rng(11)
    for shuffled in (False, True):
        _run(rt, [_task(r, nlegs, new_rank, exts, int(r.choice(nsrc)), 0.4) for _ in range(ntasks)], nlegs, new_rank, shuffled)


@pytest.mark.parametrize("nsrc", [(1,), (1, 2)], ids=["single", "several"])
def test_source_indices_past_32_bits(rt, nsrc):
    """Two source columns 2^31 elements apart (a 17 GB source)."""
    r = np.random.default_rng(12)
    tasks = []
    for _ in range(40):
        e = [int(r.integers(1, 30)), int(r.integers(1, 4)), 2]
        tasks.append((e, [1, e[0], 1], [0, 0, 1], e[0] * e[1], 2, int(r.choice(nsrc))))
    _run(rt, tasks, 3, 1, far=1 << 31)
