"""Tiled kernels at the sizes where a tile can go wrong (bit-exact against numpy)."""
import numpy as np
import pytest

from conftest import gdl

pytestmark = pytest.mark.gpu

M32 = np.uint64(0xffffffff)


def runs_of(lengths, gap=1):
    """Sorted keys whose prefixes 0, gap, 2 gap, ... have runs of these lengths."""
    lengths = np.asarray(lengths, dtype=np.int64)
    p = np.repeat(np.arange(lengths.size, dtype=np.uint64) * np.uint64(gap), lengths)
    j = np.arange(lengths.sum()) - np.repeat(np.cumsum(lengths) - lengths, lengths)
    return gdl.pack(p, j)


# a wave reads spans of 256 keys (1024 from 2^22 keys on); the last run of a
# span is followed past it, 64 keys, then doubling distances
INDEX_RUNS = {
    "one": [1], "wave": [64], "span": [256], "span+1": [257], "ends": [255, 1, 256, 2, 254, 3],
    "ones": [1] * 1025, "past64": [200, 56 + 64, 1], "past65": [200, 56 + 65, 1],
    "doubling": [1] + [255 + 64 * (1 << k) + d for k in range(6) for d in (-1, 0, 1)],
    "hub": [3, 1_000_001, 7], "mixed": [(i * i) % 97 + 1 for i in range(3000)],
    "long": [1500, 1024, 1023, 1025, 1, 4096] * 400 + [63, 64, 65] * 1500,
    "long_hub": [5, (1 << 22) + 3, 2],
}


@pytest.mark.parametrize("gap", [1, 100_003])
@pytest.mark.parametrize("name", INDEX_RUNS)
def test_index_runs_at_span_edges(ctx, name, gap):
    lengths = np.asarray(INDEX_RUNS[name], dtype=np.int64)
    keys = runs_of(lengths, gap)
    d = ctx.to_device(keys)
    idx = ctx.index_build(d, 1)
    assert idx.n_distinct == lengths.size and idx.max_run == lengths.max()
    q = np.arange(lengths.size, dtype=np.uint64) * np.uint64(gap)
    b, c = ctx.index_lookup(idx, d, q)
    assert np.array_equal(c.astype(np.int64), lengths)
    assert np.array_equal(b.astype(np.int64), np.cumsum(lengths) - lengths)
    ctx.index_free(idx)
    d.free()


def np_join_runs(inner, outer):
    p = inner >> np.uint64(32)
    lo = np.searchsorted(p, outer >> np.uint64(32))
    cnt = np.searchsorted(p, outer >> np.uint64(32), side="right") - lo
    oi = np.repeat(np.arange(outer.size), cnt)
    ii = np.repeat(lo - (np.cumsum(cnt) - cnt), cnt) + np.arange(oi.size)
    return inner[ii], outer[oi], cnt


# run lengths of the inner prefixes, and which prefix each outer tuple asks for
# (a prefix past the last one has no run): tiles are 2048 outputs, a block's
# threads take 256 outer tuples at a time
JOIN_SHAPES = {
    "one": ([1], [0]), "tile": ([2048], [0]), "tile+1": ([2048, 1], [0, 1]),
    "ends_at_tile": ([1024, 1024, 5], [0, 1, 2, 0, 1, 2]),
    "holes": ([3, 2045, 2], [9] * 300 + [0] + [9] * 700 + [1] + [9] * 5 + [2] * 2000 + [9] * 900),
    "ones": ([1] * 50, [i % 57 for i in range(5000)]),
    "hub": ([100_000, 1, 2], [1] * 10 + [0] + [2] * 600 + [7] * 600 + [0, 0, 1]),
    "words": ([63, 64, 65, 1, 128], [i % 6 for i in range(1000)]),
    "all_missing_but_last": ([4], [5] * 3000 + [0]),
    # enough tiles for a block to take several
    "many": ([i % 40 for i in range(1, 4000)], [(i * 7919) % 4100 for i in range(600_000)]),
}


def some(n, hits, prefixes, at=None):
    """n outer tuples of which `hits` find one of `prefixes` runs, the others none."""
    rng = np.random.default_rng(n + hits)
    asks = np.full(n, prefixes + 7)
    asks[rng.choice(n, hits, replace=False) if at is None else at] = \
        rng.integers(0, prefixes, hits)
    return asks


# fewer outputs than outer tuples: each thread searches for the owner of the
# first of its 1, 2 or 4 consecutive outputs (up to 2^18 outputs; up to 2^20 or
# a quarter of the outer tuples; above), tiles of 256 of those
JOIN_SHAPES.update({
    "sparse_one": ([1], some(5000, 1, 1, [4999])), "sparse_first": ([1], some(5000, 1, 1, [0])),
    "sparse_255": ([1], some(9000, 255, 1)), "sparse_256": ([1], some(9000, 256, 1)),
    "sparse_257": ([1], some(9000, 257, 1)), "sparse_ends": ([256, 1, 2], some(4000, 9, 3)),
    "sparse_block": ([1], some(70_000, 300, 1, np.arange(65_000, 65_300))),
    "sparse_hub": ([90_000, 1, 3], some(200_000, 3, 3)),
    "sparse_runs": ([(i * 7) % 23 for i in range(500)], some(100_000, 4000, 500)),
    "sparse_2^18": ([1], some(300_000, 1 << 18, 1)),
    "sparse_two": ([1], some(300_000, (1 << 18) + 1, 1)),
    "sparse_two_runs": ([3, 1, 8, 2], some(400_000, 99_999, 4)),
    "sparse_2^20": ([1], some(1_100_000, 1 << 20, 1)),
    "sparse_four": ([1], some(1_100_000, (1 << 20) + 1, 1)),
    "sparse_four_runs": ([9, 1, 40], some(2_000_000, 70_000, 3)),
    "sparse_quarter": ([1, 2], some(5_000_000, 750_000, 2)),
    "as_many_as_outer": ([2], some(200_000, 100_000, 1)),
})


@pytest.mark.parametrize("name", JOIN_SHAPES)
def test_join_outputs_at_tile_edges(ctx, name):
    lengths, asks = JOIN_SHAPES[name]
    inner = runs_of(lengths)
    outer = gdl.pack(np.asarray(asks), np.arange(len(asks)))
    ik, ok, _ = np_join_runs(inner, outer)
    got = ctx.join(inner, outer, (1, 3))  # (inner c1, outer c1)
    assert np.array_equal(got, ((ik & M32) << np.uint64(32)) | (ok & M32))


# outputs that few of the outer tuples have take less time than outputs of all
def test_join_time_where_most_outer_tuples_miss(ctx):
    inner, n = runs_of([8] * 50_000), 2_000_000

    def ms(hits):
        outer = gdl.pack(some(n, hits, 50_000), np.arange(n))
        best = 1e9
        for _ in range(3):
            ctx.stats_reset()
            ctx.join(inner, outer, (1, 3))
            best = min(best, ctx.stats()["join_materialize"]["total_ms"])
        return best

    ctx.stats_enable(True)
    try:
        assert ms(200) < ms(n)
    finally:
        ctx.stats_enable(False)
        ctx.stats_reset()


def _sorted(rng, n, hi):
    return np.sort(rng.choice(hi, size=n, replace=False)).astype(np.uint64) if n else \
        np.zeros(0, np.uint64)


# tiles are 2048 keys of the merged sequence, 8192 from 2^19 on; a tile may hold
# one side only, and a duplicate may be the first key of a tile
BIG = 1 << 18
@pytest.mark.parametrize("na,nb,hi", [
    (0, 1, 9), (1, 0, 9), (1, 1, 1), (2047, 1, 5000), (1024, 1024, 2048), (1024, 1024, 1024),
    (2048, 2048, 2048), (2049, 2047, 4097), (5000, 5000, 5500), (100_000, 10, 10**6),
    (10, 100_000, 10**6), (300_001, 299_999, 600_000), (700_000, 700_000, 700_000),
    (BIG, BIG - 1, 2 * BIG), (BIG, BIG, BIG), (BIG + 4096, BIG + 4095, 600_000),
    (BIG + 4096, BIG + 4096, BIG + 4096), (BIG + 4097, BIG + 4096, 600_000),
    (2 * BIG + 8192, 1, 600_000), (1, 2 * BIG + 8192, 600_000)])
def test_merge_at_tile_edges(ctx, na, nb, hi):
    rng = np.random.default_rng(na * 7 + nb)
    a, b = _sorted(rng, na, hi), _sorted(rng, nb, hi)
    for full, newt in ((a, b), (a, b + np.uint64(hi)), (a + np.uint64(hi), b)):
        u, d = ctx.merge_diff(full, newt)
        assert np.array_equal(u, np.union1d(full, newt))
        assert np.array_equal(d, np.setdiff1d(newt, full))
        assert np.array_equal(ctx.merge_union(full, newt), u)
        assert np.array_equal(ctx.set_difference(newt, full), d)


def test_tile_words_are_tagged_anew(ctx):
    # the running sums' words are cleared once in 255 calls and tagged in between
    a = np.arange(0, 60_000, 2, dtype=np.uint64)
    for i in range(600):
        n = 5000 + 97 * (i % 300)
        b = np.arange(i % 7, 3 * n, 3, dtype=np.uint64)
        assert ctx.set_difference(b, a).size == np.setdiff1d(b, a, assume_unique=True).size


# tiles of 4096 keys, of 16384 from 2^20 keys on
@pytest.mark.parametrize("n", [1, 63, 64, 65, 4095, 4096, 4097, 12_289, (1 << 20) - 1, 1 << 20,
                               (1 << 20) + 1, (1 << 20) + 16_383, (1 << 20) + 16_385, 2_000_003])
@pytest.mark.parametrize("kind", ["none", "all", "half", "last", "tile_firsts"])
def test_compaction_at_tile_edges(ctx, n, kind):
    i = np.arange(n)
    keep = {"none": i < 0, "all": i >= 0, "half": i % 2 == 1, "last": i == n - 1,
            "tile_firsts": i % (4096 if n < 1 << 20 else 16_384) == 0}[kind]
    # c0 == 7 where kept (a predicate on a column), c1 tells the keys apart
    keys = gdl.pack(np.where(keep, 7, 8), i)
    assert np.array_equal(ctx.filter(keys, gdl.PRED_EQ | 0x100, 0, 7), keys[keep])


# what a compaction reads, and the keys it keeps
@pytest.mark.parametrize("n,kept", [(1000, 1), (50_000, 50_000), (1_200_000, 240_000)])
def test_compaction_counts_the_bytes_it_moves(ctx, n, kept):
    keys = (np.arange(n) // (n // kept)).astype(np.uint64)
    ctx.stats_reset()
    assert ctx.unique(keys).size == kept
    s = ctx.stats()["compact"]
    ctx.stats_reset()
    assert s["launches"] == 1 and s["alg_bytes"] == 8 * (n + kept)


# one launch up to 2^22 values, three above; 2048 values a tile, 8192 from 2^18 on
SCAN_SIZES = [1, 8, 2047, 2048, 2049, 100_000, BIG - 1, BIG, BIG + 1, BIG + 8191, BIG + 8193,
              1 << 22, (1 << 22) + 1]


# a join's run starts and their scan: the same sizes of the outer relation
@pytest.mark.parametrize("n", SCAN_SIZES)
def test_join_offsets_at_tile_edges(ctx, n):
    lengths = [i % 4 for i in range(1000)]
    inner = runs_of(lengths)
    outer = gdl.pack((np.arange(n) * 7919) % 1009, np.arange(n))
    ik, ok, _ = np_join_runs(inner, outer)
    got = ctx.join(inner, outer, (1, 3))
    assert np.array_equal(got, ((ik & M32) << np.uint64(32)) | (ok & M32))


@pytest.mark.parametrize("n", SCAN_SIZES)
def test_scan_at_tile_edges(ctx, n):
    import ctypes
    counts = (np.arange(n, dtype=np.uint64) * np.uint64(2654435761) & M32).astype(np.uint32)
    counts[::3] = 0
    d, o = ctx.to_device(counts, np.uint32), ctx.alloc(n + 1)
    total = ctypes.c_uint64()
    ctx._check(ctx.eng.gdl_join_scan(ctx.h, d.ptr, n, o.ptr, ctypes.byref(total)), "scan")
    want = np.concatenate([[0], np.cumsum(counts.astype(np.uint64))]).astype(np.uint64)
    assert np.array_equal(o.numpy(), want) and total.value == int(want[-1])
    d.free(); o.free()


# tiles of 2048 keys up to 2^18 keys, of 4096 up to 2^20, of 8192 above
@pytest.mark.parametrize("n", [4097, 6144, (1 << 18) - 1, 1 << 18, (1 << 18) + 1, 1 << 20,
                               (1 << 20) + 1, 1_100_003, 1 << 22, (1 << 22) + 8193])
@pytest.mark.parametrize("kind", ["random36", "random32", "sorted", "reversed", "one_odd",
                                  "few", "high_only"])
def test_sort_at_tile_edges(ctx, n, kind):
    rng = np.random.default_rng(n)
    i = np.arange(n, dtype=np.uint64)
    bits = 18 if kind == "random36" else 16 if kind == "random32" else 32
    if kind.startswith("random"):
        keys = gdl.pack(rng.integers(0, 1 << bits, n), rng.integers(0, 1 << bits, n))
    elif kind == "one_odd":
        keys = np.full(n, 0x0102030405060708, dtype=np.uint64)
        keys[n // 2] = 0x0102030405060701
    else:
        keys = {"sorted": i * np.uint64(977), "reversed": i[::-1] * np.uint64(977),
                "few": (i * np.uint64(7919)) % np.uint64(3) << np.uint64(40),
                "high_only": gdl.pack(rng.integers(0, 1 << 31, n), np.zeros(n))}[kind]
    assert np.array_equal(ctx.sort(keys, bits, bits), np.sort(keys))
    assert np.array_equal(ctx.sort_unique(keys, -1, -1), np.unique(keys))


# a linear body's blocks hand over their counts packed in one word up to 2^27
# produced tuples and 1023 blocks (of 256 outer tuples up to 2^16 of them, of
# 512 above), in words of their own above; the ids need a hash set
@pytest.mark.parametrize("paths", [1, 1023, 1025, 21_845, 21_846, 174_592, 174_593, 400_000,
                                   1_200_000])
def test_linear_bodies_of_disjoint_paths(ctx, paths):
    # node j of path i is i + j * paths + 2^19: three edges a path, in any order
    i = np.arange(paths, dtype=np.uint64) + np.uint64(1 << 19)
    node = [i + np.uint64(j * paths) for j in range(4)]
    edges = np.concatenate([gdl.pack(node[j], node[j + 1]) for j in (1, 0, 2)])
    got = ctx.run_tc(edges, out_cap=8 * paths)
    want = np.sort(np.concatenate([gdl.pack(node[a], node[b])
                                   for a in range(4) for b in range(a + 1, 4)]))
    assert np.array_equal(got["out"], want)
    assert [t[3] for t in got["trace"]] == [2 * paths, paths, 0]
    assert [t[2] for t in got["trace"]] == [2 * paths, paths, 0]


# with runs of up to 1000 the limit of 2^27 produced tuples is a delta of
# 134,217: first deltas on both sides of it, and one that grows past it
@pytest.mark.parametrize("first", [134_216, 134_217, 134_218, 1200])
def test_linear_bodies_around_the_packed_limit(ctx, first):
    base, ins, outs = 1 << 19, np.arange(1000), np.arange(100 if first > 1200 else 200)
    hub, extra = 0, np.arange(first - ins.size - outs.size)
    into = gdl.pack(base + 1 + ins, np.full(ins.size, base + hub))
    out = gdl.pack(np.full(outs.size, base + hub), base + 5000 + outs)
    alone = gdl.pack(base + 10_000 + 2 * extra, base + 10_001 + 2 * extra)
    edges = np.concatenate([into, out, alone])
    pairs = gdl.pack(np.repeat(base + 1 + ins, outs.size), np.tile(base + 5000 + outs, ins.size))
    got = ctx.run_tc(edges, out_cap=edges.size + pairs.size)
    assert np.array_equal(got["out"], np.sort(np.concatenate([edges, pairs])))
    assert [t[3] for t in got["trace"]] == [pairs.size, 0]
    assert [t[2] for t in got["trace"]] == [pairs.size, 0]


# a result of n keys goes straight into a buffer that holds it; a smaller one
# is refused and left as it was
@pytest.mark.parametrize("prog", ["tc", "sg", "path_length"])
@pytest.mark.parametrize("short", [0, 1])
def test_program_results_into_the_callers_buffer(ctx, prog, short):
    import ctypes
    e = gdl.gen_er(7, 300, 900)
    fn = {"tc": ctx.run_tc, "sg": ctx.run_sg, "path_length": ctx.run_path_length}[prog]
    want = fn(e)
    n = want["n_out"]
    p64, p32 = ctypes.POINTER(ctypes.c_uint64), ctypes.POINTER(ctypes.c_uint32)
    out = np.full(n + 8, 5, dtype=np.uint64)
    lens = np.full(n + 8, 5, dtype=np.uint32)
    res = gdl.ProgResult()
    src = e.ctypes.data_as(ctypes.c_void_p)
    if prog == "path_length":
        st = ctx.prog.gdl_prog_path_length(ctx.h, src, e.size, 0, ctypes.byref(res),
                                           out.ctypes.data_as(p64), lens.ctypes.data_as(p32),
                                           n - short)
    else:
        b = gdl.ProgBuffers()
        b.out, b.out_cap = out.ctypes.data_as(p64), n - short
        args = (ctx.h, src, e.size, 0) + ((-1,) if prog == "tc" else ())
        st = getattr(ctx.prog, "gdl_prog_" + prog)(*args, ctypes.byref(res), ctypes.byref(b))
    assert st == (5 if short else 0) and res.n_out == n
    k = 0 if short else n
    assert np.array_equal(out[:k], want["out"][:k]) and np.all(out[k:] == 5)
    if prog == "path_length":
        assert np.array_equal(lens[:k], want["lens"][:k]) and np.all(lens[k:] == 5)


# a recorded sort replays with other keys and after other sorts
@pytest.mark.parametrize("n", [4097, 300_000, 1_100_003])
def test_sort_in_a_graph(ctx, n):
    ctx.stats_enable(False)
    rng = np.random.default_rng(n)
    sets = [gdl.pack(rng.integers(0, 1 << 18, n), rng.integers(0, 1 << 18, n)) for _ in range(4)]
    d, o = ctx.to_device(sets[0]), ctx.alloc(n)

    def sort():
        ctx._check(ctx.eng.gdl_sort_u64(ctx.h, d.ptr, n, 18, 18, o.ptr), "sort")

    sort()  # the scratch is in the context's pool from here on
    ctx.sync()
    ctx.graph_begin()
    sort()
    g = ctx.graph_end()
    for k in sets + sets[:1]:
        assert np.array_equal(ctx.sort(k[: n // 2 + 4096]), np.sort(k[: n // 2 + 4096]))
        ctx._check(ctx.eng.gdl_memcpy_h2d(ctx.h, d.ptr, k.ctypes.data, k.nbytes), "h2d")
        ctx.graph_launch(g)
        ctx.sync()
        assert np.array_equal(o.numpy(), np.sort(k))
    ctx.graph_destroy(g)
    d.free(); o.free()


# recorded sorts share one set of digit counts: two in one graph, and two graphs
# in turn, with a sort between
def test_recorded_sorts_take_turns(ctx):
    ctx.stats_enable(False)
    rng = np.random.default_rng(3)
    sizes = [5000, 300_000, 40_000]
    d, o = [ctx.alloc(n) for n in sizes], [ctx.alloc(n) for n in sizes]

    def sort(i):
        ctx._check(ctx.eng.gdl_sort_u64(ctx.h, d[i].ptr, sizes[i], 18, 18, o[i].ptr), "sort")

    for i in range(3):
        sort(i)
    ctx.sync()
    graphs = []
    for which in ((0, 1), (2,)):
        ctx.graph_begin()
        for i in which:
            sort(i)
        graphs.append(ctx.graph_end())
    for _ in range(4):
        keys = [gdl.pack(rng.integers(0, 1 << 18, n), rng.integers(0, 1 << 18, n)) for n in sizes]
        for i in range(3):
            ctx._check(ctx.eng.gdl_memcpy_h2d(ctx.h, d[i].ptr, keys[i].ctypes.data,
                                              keys[i].nbytes), "h2d")
        ctx.graph_launch(graphs[0])
        ctx.graph_launch(graphs[1])
        assert np.array_equal(ctx.sort(keys[1], 18, 18), np.sort(keys[1]))
        for i in range(3):
            assert np.array_equal(o[i].numpy(), np.sort(keys[i]))
    for g in graphs:
        ctx.graph_destroy(g)
    for x in d + o:
        x.free()


# a block takes 4096 slots a round, the last round holds the word of the key ~0
@pytest.mark.parametrize("n", [0, 1, 700, 5000, 300_000])
@pytest.mark.parametrize("top", [False, True])
def test_set_extraction_by_blocks(ctx, n, top):
    keys = np.unique(np.random.default_rng(n).integers(0, 1 << 63, n, dtype=np.uint64))
    if top:
        keys = np.append(keys, np.uint64(0xffffffffffffffff))
    hs = ctx.hashset_create(0)
    if keys.size:
        assert ctx.hashset_insert_new(hs, keys).size == keys.size
    assert np.array_equal(np.sort(ctx.hashset_extract(hs)), keys)
    ctx.hashset_free(hs)
