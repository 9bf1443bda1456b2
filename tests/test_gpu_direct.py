"""GPU tests of the direct range kernel (csrc/direct.hip) at the edges of its lists and tables:
K+1 around the sizes its three builds end at (40, 224, 448), point counts around a wave and a
chunk, blocks from empty to crowded, equal keys and equal coordinates, root arguments below the
fast path's range.  Rows are compared with FP64 brute force (ids, and FP32 distance bits)."""
import numpy as np
import pytest

from hybrid_k_nearest_neighbor_self_join_amd import _lib, batched, learned_radius, synthetic

pytestmark = pytest.mark.gpu


def _check(oracle, pts, k, **kw):
    ids, dist, st = _lib.knnjoin_ex(pts, k, brute_fallback=0, **kw)
    perm, _ = oracle.reorder(pts)
    bi, bd = oracle.bruteforce(np.ascontiguousarray(pts[:, perm]), k)
    assert np.array_equal(ids, bi)
    assert np.array_equal(dist.view(np.uint32), bd.view(np.uint32))
    return st


@pytest.mark.parametrize("k", [1, 38, 39, 40, 63, 64, 127, 128, 191, 223, 224, 300, 447, 448])
def test_list_sizes(oracle, k):
    st = _check(oracle, synthetic.mixed_box(6007, seed=k), k, beta=0.025)
    assert st.overflow_queries == 0


@pytest.mark.parametrize("n", [2, 63, 64, 65, 129, 4097])
@pytest.mark.parametrize("d,nd", [(1, 1), (2, 2), (3, 2), (3, 3), (5, 4), (6, 5), (8, 6), (9, 7)])
def test_point_counts_and_dims(oracle, n, d, nd):
    pts = np.random.default_rng(n * 10 + d).uniform(-3.0, 5.0, (n, d)).astype(np.float32)
    _check(oracle, pts, min(5, n - 1), num_indexed_dims=nd, beta=0.05)


@pytest.mark.parametrize("mode", [_lib.KNN_MODE_BETA, _lib.KNN_MODE_LEARNED])
def test_crowded_and_empty_blocks(oracle, mode):
    # one dense cluster (blocks of thousands of points: shrunk radii, tightened lists), a sparse
    # background and far outliers (many passes)
    learned_radius.register_default_models()
    rng = np.random.default_rng(5)
    pts = np.concatenate([rng.normal(0.0, 0.01, (6000, 2)), rng.uniform(-50, 50, (3000, 2)),
                          rng.uniform(400, 500, (5, 2))]).astype(np.float32)
    _check(oracle, pts[rng.permutation(len(pts))], 20, mode=mode)


@pytest.mark.parametrize("d,nd", [(2, 2), (3, 3), (4, 2)])
def test_equal_keys(oracle, d, nd):
    # a coarse lattice: every distance is shared by many points, ranked by id
    rng = np.random.default_rng(d)
    pts = (rng.integers(0, 24 if d == 2 else 8, (5000, d)) / 8.0).astype(np.float32)
    _check(oracle, pts, 30, num_indexed_dims=nd, beta=0.025)


@pytest.mark.parametrize("scale", [1e-18, 3e-17, 1e-10])
def test_small_distances(oracle, scale):
    # squared distances around and below 2^-96, where the root needs its scaled form
    pts = (np.random.default_rng(3).uniform(0, 1, (3000, 2)) * scale).astype(np.float32)
    _check(oracle, pts, 8)


def test_double_rows(oracle):
    pts = np.random.default_rng(9).uniform(0, 1, (5000, 3))
    ids, dist, _ = _lib.knnjoin_ex(pts, 24, brute_fallback=0)
    perm, _ = oracle.reorder(pts)
    bi, bd = oracle.bruteforce(np.ascontiguousarray(pts[:, perm]), 24)
    assert np.array_equal(ids, bi)
    assert np.array_equal(dist.view(np.uint64), bd.view(np.uint64))


@pytest.mark.parametrize("d,nd,k,dtype,mode", [
    (3, 1, 8, np.float32, "plain"), (4, 2, 40, np.float64, "plain"), (6, 4, 16, np.float32, "plain"),
    (6, 1, 5, np.float32, "plain"), (9, 3, 16, np.float32, "plain"), (16, 2, 4, np.float64, "plain"),
    (7, 7, 8, np.float32, "plain"), (4, 2, 16, np.float32, "learned"), (6, 4, 33, np.float64, "learned"),
    (6, 4, 450, np.float32, "learned"),
])
@pytest.mark.parametrize("data", ["mixed", "flat", "far"])
def test_grid_dims(oracle, monkeypatch, d, nd, k, dtype, mode, data):
    # a grid over more dims than the join indexes gives the rows, the schedule and the failures of
    # the indexed dims' grid: "flat" has constant dims, "far" one whose cells do not fit a table
    rng = np.random.default_rng(7 * d + nd)
    n = 6000
    pts = rng.random((n, d))
    pts[n // 2:] = 0.5 + 0.01 * rng.normal(size=(n - n // 2, d))
    pts[100:140] = pts[100]
    if data == "flat":
        pts[:, nd:] = 0.25
    if data == "far":
        pts *= 0.5 ** np.arange(d)  # the indexed dims are those of the largest variance
        pts[0] *= 10.0
    pts = pts.astype(dtype)
    if mode == "learned":
        learned_radius.register_default_models()
    m = _lib.KNN_MODE_LEARNED if mode == "learned" else _lib.KNN_MODE_BETA
    res = []
    for dims in ("0", "6"):
        monkeypatch.setenv("KNN_GRID_DIMS", dims)
        res.append(_lib.knnjoin_ex(pts, k, num_indexed_dims=nd, mode=m, brute_fallback=0))
    (i0, d0, s0), (i1, d1, s1) = res
    perm, _ = oracle.reorder(pts)
    q = rng.choice(n, 300, replace=False)
    bi, bd = oracle.bruteforce(np.ascontiguousarray(pts[:, perm]), k, queries=q)
    assert np.array_equal(i1[q], bi) and np.array_equal(d1[q], bd)
    assert np.array_equal(i0, i1) and np.array_equal(d0, d1)
    if mode == "plain":
        assert (s0.iterations, s0.reindexes, s0.eps0, s0.eps_final) == (s1.iterations, s1.reindexes, s1.eps0, s1.eps_final)


@pytest.mark.parametrize("d,gen", [(2, "mixed"), (2, "uniform"), (4, "uniform"), (6, "skewed")])
@pytest.mark.parametrize("k", [455, 479, 495, 496])
def test_longest_lists(oracle, d, gen, k):
    # K+1 up to 496: the direct kernel; 497: the collect kernel.  A batched join reports the tile
    # size of the kernel it takes
    n = 8009
    pts = {"mixed": synthetic.mixed_box, "uniform": lambda n, seed: synthetic.unit_cube(n, d, seed=seed),
           "skewed": lambda n, seed: synthetic.skewed_cube(n, d, seed=seed)}[gen](n, seed=k)
    _check(oracle, pts, k, beta=0.025)
    assert batched.knnjoin_batched([pts], [k])[2].tile_queries == (64 if k < 496 else 16)


@pytest.mark.parametrize("kern", ["direct", "collect"])
@pytest.mark.parametrize("n", [7, 65, 500, 9001])
def test_tile_ranges(oracle, monkeypatch, kern, n):
    # one queue over all tiles or one range per XCD, with fewer tiles than ranges and with many:
    # every tile is taken once whichever range it lies in
    monkeypatch.setenv("KNN_RANGE_KERNEL", kern)
    pts = synthetic.skewed_cube(n, 3, seed=n)
    cand = set()
    for ranges in ("1", "8"):
        monkeypatch.setenv("KNN_TILE_RANGES", ranges)
        cand.add(_check(oracle, pts, min(5, n - 1), beta=0.05).candidates)
    assert len(cand) == 1


@pytest.mark.parametrize("div", ["1", "2", "2.5", "4.5", "5", "6"])
def test_rows_looked_up_together(oracle, monkeypatch, div):
    # blocks of 2 div to 2 div + 2 rows (a chunk's table holds 10: at 4.5 some and at 5 most blocks
    # have more, and are streamed), looked up one or two at a time
    monkeypatch.setenv("KNN_PLAIN_GRID_DIV", div)
    monkeypatch.setenv("KNN_PLAIN_MAX_REACH", div)
    pts = synthetic.mixed_box(9001, seed=int(10 * float(div)))
    st = [_check(oracle, pts, 20, beta=0.025)]
    monkeypatch.setenv("KNN_TILE_ROWS", "1")
    st.append(_check(oracle, pts, 20, beta=0.025))
    assert st[0].candidates == st[1].candidates and st[0].iterations == st[1].iterations


@pytest.mark.parametrize("ranges", ["1", "8"])
@pytest.mark.parametrize("grid", [1, 5, 9, 100, 4096])
def test_first_tiles(monkeypatch, ranges, grid):
    # every workgroup has a first tile of its own and takes the rest from the queues: fewer workgroups
    # than ranges, uneven shares of them, more workgroups than tiles
    monkeypatch.setenv("KNN_TILE_RANGES", ranges)
    sets = [synthetic.skewed_cube(n, d, seed=n) for n, d in ((3, 2), (700, 2), (1, 3), (2500, 3), (65, 6))]
    ks = [2, 9, 0, 12, 5]
    for kern in ("direct", "collect"):
        monkeypatch.setenv("KNN_RANGE_KERNEL", kern)
        ids, dists, st = batched.knnjoin_batched(sets, ks, grid_blocks=grid, tile_queries=16)
        for p, k, i, d in zip(sets, ks, ids, dists):
            ri, rd, _ = _lib.knnjoin_ex(p, k, brute_fallback=0)
            assert np.array_equal(i, ri) and np.array_equal(d.view(np.uint32), rd.view(np.uint32))


@pytest.mark.parametrize("ranges", ["1", "8"])
@pytest.mark.parametrize("n", [2101, 3000])
def test_first_tiles_of_the_heap_kernel(oracle, monkeypatch, ranges, n):
    monkeypatch.setenv("KNN_TILE_RANGES", ranges)
    _check(oracle, synthetic.skewed_cube(n, 3, seed=n), 2100, beta=0.05)
