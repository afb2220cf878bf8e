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


def block(nbytes):
    """The allocator's block for a request of a call's scratch."""
    nbytes += 16
    step = 1 << max(nbytes.bit_length() - 4, 0)
    return 512 if nbytes <= 512 else -(-nbytes // step) * step


# A sort of n keys fits room for a second buffer of them, a count per digit (9
# bits) and 4096 keys, and the digits' totals (and an eighth of the counts, the
# step of the allocator's blocks).
def sort_room(n):
    counts = 4 * 512 * -(-n // 4096)
    return block(8 * n) + block(counts) + counts // 8 + block(4 * 512)


@pytest.mark.parametrize("n", [4097, 12_289, 100_000, 1 << 18, (1 << 18) + 1, 700_001, 1 << 20,
                               1_500_000])
def test_sort_in_little_scratch(ctx, n):
    keys = gdl.pack(*np.random.default_rng(n).integers(0, 1 << 18, (2, n)))
    d, o = ctx.to_device(keys), ctx.alloc(n)
    ctx.release_cached()
    ctx.set_mem_cap(ctx.mem_info()["in_use"] + sort_room(n))
    try:
        for _ in range(2):
            ctx._check(ctx.eng.gdl_sort_u64(ctx.h, d.ptr, n, 18, 18, o.ptr), "sort")
    finally:
        ctx.set_mem_cap(0)
    assert np.array_equal(o.numpy(), np.sort(keys))
    d.free(); o.free()


# From 2^30 keys on a tile's digit counts take 64-bit words (tiles of 16384
# keys); the recorded form replays with other keys.
@pytest.mark.parametrize("recorded", [False, True])
def test_sort_of_more_than_2_to_the_30_keys(ctx, recorded):
    torch = pytest.importorskip("torch")
    n = (1 << 30) + 12_345
    if torch.cuda.mem_get_info()[0] < 120 << 30:
        pytest.skip("needs 120 GB of device memory")
    ctx.stats_enable(False)
    ctx.release_cached()
    keys = torch.empty(n, dtype=torch.int64, device="cuda")
    out = torch.empty_like(keys)

    def draw(seed):
        g = torch.Generator(device="cuda").manual_seed(seed)
        torch.randint(0, 1 << 36, (n,), device="cuda", generator=g, out=keys)
        keys.copy_(((keys >> 18) << 32) | (keys & 0x3ffff))
        out.zero_()
        torch.cuda.synchronize()

    def sort():
        ctx._check(ctx.eng.gdl_sort_u64(ctx.h, keys.data_ptr(), n, 18, 18, out.data_ptr()), "sort")

    def right():
        ctx.sync()
        return bool(torch.equal(out, torch.sort(keys)[0]))

    draw(1)
    ctx.set_mem_cap(ctx.mem_info()["in_use"] + sort_room(n))
    try:
        sort()
    finally:
        ctx.set_mem_cap(0)
    assert right()
    if recorded:
        ctx.graph_begin()
        sort()
        g = ctx.graph_end()
        for seed in (2, 3):
            draw(seed)
            ctx.graph_launch(g)
            assert right()
        ctx.graph_destroy(g)
    del keys, out
    torch.cuda.empty_cache()
    ctx.release_cached()
