"""Calls at the edge of a context's byte cap: what fits is not refused."""
import ctypes

import numpy as np
import pytest

from conftest import gdl

pytestmark = pytest.mark.gpu

u64 = ctypes.c_uint64


def paths(n):
    """n disjoint paths of three edges over ids from 2^19 on; the edges, and the closure."""
    i = np.arange(n, dtype=np.uint64) + np.uint64(1 << 19)
    node = [i + np.uint64(j * n) for j in range(4)]
    pairs = [gdl.pack(node[a], node[b]) for a in range(4) for b in range(a + 1, 4)]
    return (np.sort(np.concatenate([gdl.pack(node[j], node[j + 1]) for j in range(3)])),
            np.sort(np.concatenate(pairs)))


# The log has room for every body (3n edges, then 2n and n new tuples, a body's
# room checked ahead of it) and none to spare is left under the cap: a larger
# log, or scratch beyond the loop's state and its bodies' counts, is refused.
@pytest.mark.parametrize("n", [3000, 20_000, 200_000])
def test_linear_fixpoint_in_the_log_it_has(ctx, n):
    fn = ctx.eng.gdl_fixpoint_linear
    fn.restype = ctypes.c_int
    pu = ctypes.POINTER(u64)
    fn.argtypes = [ctypes.c_void_p, ctypes.c_void_p, u64, ctypes.POINTER(gdl.Index), gdl.ColMap,
                   gdl.Pred, ctypes.POINTER(gdl.HashSet), ctypes.POINTER(ctypes.c_void_p), pu, pu,
                   pu, ctypes.c_int, pu, pu, ctypes.POINTER(ctypes.c_int)]
    edges, closure = paths(n)
    swapped = np.sort((edges >> np.uint64(32)) | (edges << np.uint64(32)))
    cap = 8 * n
    inner, log, fresh = ctx.to_device(swapped), ctx.alloc(cap), ctx.alloc(edges.size)
    ctx._check(ctx.eng.gdl_memcpy_h2d(ctx.h, log.ptr, edges.ctypes.data, edges.nbytes), "h2d")
    idx = ctx.index_build(inner, 1)
    hs = ctx.hashset_create(40 * n + 16_384)
    m = u64()
    ctx._check(ctx.eng.gdl_hashset_insert_new(ctx.h, ctypes.byref(hs), log.ptr, edges.size,
                                              fresh.ptr, ctypes.byref(m)), "insert")
    tc = gdl.ColMap(2, (ctypes.c_int32 * 2)(gdl.COL_INNER1, gdl.COL_OUTER1))
    at, room, begin, end = ctypes.c_void_p(log.ptr), u64(cap), u64(0), u64(edges.size)
    new, raw, bodies = np.zeros(8, np.uint64), np.zeros(8, np.uint64), ctypes.c_int()
    ctx.set_mem_cap(ctx.mem_info()["in_use"] + 8192)
    try:
        st = fn(ctx.h, inner.ptr, inner.n, ctypes.byref(idx), tc, gdl.Pred(gdl.PRED_NONE, 0, 1),
                ctypes.byref(hs), ctypes.byref(at), ctypes.byref(room), ctypes.byref(begin),
                ctypes.byref(end), 8, gdl._p64(new), gdl._p64(raw), ctypes.byref(bodies))
    finally:
        ctx.set_mem_cap(0)
    log.ptr = at.value
    assert st == 0 and room.value == cap and end.value == closure.size
    assert bodies.value == 3 and list(new[:3]) == [2 * n, n, 0]
    assert np.array_equal(np.sort(log.numpy(closure.size)), closure)
    ctx.index_free(idx)
    ctx.hashset_free(hs)
    for x in (inner, log, fresh):
        x.free()


# More than 16384 tiles of a merge take their running sums' words from the
# pool: the byte cap counts them, and a call that they fit gives the same result.
def test_tile_words_of_a_large_merge_are_counted(ctx):
    n = (1 << 27) + 1000
    full = np.arange(n, dtype=np.uint64) * np.uint64(2)
    newt = np.concatenate([full[:: n // 7], full[:: n // 5] + np.uint64(1), full[-1:]])
    newt = np.unique(newt)
    f, t, d = ctx.to_device(full), ctx.to_device(newt), ctx.alloc(newt.size)
    m = u64()

    def diff(room):
        ctx.set_mem_cap(ctx.mem_info()["in_use"] + room)
        try:
            return ctx.eng.gdl_set_difference_u64(ctx.h, t.ptr, newt.size, f.ptr, n, d.ptr,
                                                  ctypes.byref(m))
        finally:
            ctx.set_mem_cap(0)

    want = newt[newt % np.uint64(2) == 1]
    assert diff(1 << 16) == 2  # the words of 16385 tiles are 131 kB
    for _ in range(3):
        m.value = 0
        assert diff(1 << 20) == 0 and np.array_equal(d.numpy(m.value), want)
    for x in (f, t, d):
        x.free()
