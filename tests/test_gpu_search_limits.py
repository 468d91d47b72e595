"""The search at the limits of its staged boxes' arithmetic: clouds whose cells are
tiny beside their coordinates, or whose distances leave FP32's range when
squared, at row counts that leave lanes of the last wave without a query.  Lists
hold the oracle's KD3 neighbors, and feature columns and statuses equal the
growing search's, bit for bit, for a cloud and a batch."""
import numpy as np
import pytest

import gpupdal_amd as g
from helpers import set_equal_rows
from test_gpu_search_paths import cloud as path_cloud

pytestmark = pytest.mark.gpu


def cloud(kind, n):
    rng = np.random.default_rng(n)
    if kind == "coincident":  # one place, at negative y
        p = np.tile([1.0, -5.0, 0.0], (n, 1))
    elif kind == "millimetres":  # a fine scan in geocentric coordinates
        p = rng.uniform(0, 1, (n, 3)) * [0.02, 0.02, 0.002] + [5e5, -4e6, -3e6]
    elif kind == "tall":  # neighbors farther than the search's largest radius
        p = rng.uniform(0, 1, (n, 3)) * [10.0, 10.0, 1.5 * n]
    elif kind.startswith("scale"):  # spacings at and beyond the FP32 keys' range
        p = rng.normal(size=(n, 3)) * float(kind[5:])
    else:  # "corner": all coordinates large and negative
        p = rng.uniform(0, 1, (n, 3)) * [1e-3, 1e-3, 1e-3] - 6.4e6
    return np.ascontiguousarray(p.T)


def same_bits(a, b):
    assert np.array_equal(a[1][0], b[1][0])
    for ca, cb in zip(a[0][0], b[0][0]):
        assert np.array_equal(np.asarray(ca).view(np.uint64), np.asarray(cb).view(np.uint64))


@pytest.mark.parametrize("k", [1, 8, 9, 20, 36, 40])
@pytest.mark.parametrize("n", [63, 65, 100, 333])
@pytest.mark.parametrize("kind", ["coincident", "millimetres", "corner", "tall", "scale1e17", "scale1e18",
                                  "scale1e20", "scale1e40", "scale1e-12", "scale1e-21"])
def test_limits(oracle, kind, n, k):
    x, y, z = cloud(kind, n)
    c, slow = g.Context(0), g.Context(0)
    slow.set_tuning("set_select", 0)
    cl = c.cloud(x, y, z)
    ids, _ = cl.knn(k)
    # (the oracle's lists are KD3Index's, so rows of coincident points agree too)
    assert set_equal_rows(ids, oracle.kd3(x, y, z).neighbors_all(k, threads=4)).all()
    st = [g.stage(g.STAGE_COVFEAT, k + 2, features=g.F_ALL10)]
    want = slow.cloud(x, y, z).run(st, init=np.nan)
    same_bits(cl.run(st, init=np.nan), want)
    b = c.batch([(x, y, z), (x[:50], y[:50], z[:50])])
    got = b.run(st, init=np.nan)
    same_bits(([[b.tile(col, 0) for col in got[0][0]]], [b.tile(got[1][0], 0)]), want)
    b.close()
    slow.close()
    c.close()


@pytest.mark.parametrize("n", [4, 5, 17, 32767, 32769, 131071, 131072, 131080, 200003])
def test_growing_search_row_counts(n):
    # Every row by the growing search, at counts beside the waves' first rows,
    # the lists held together and the larger draws: the same columns, statuses
    # and lists as the query-per-lane search.
    rng = np.random.default_rng(n)
    x, y, z = np.ascontiguousarray((rng.uniform(0, 1, (n, 3)) * [n ** 0.5, n ** 0.5, 1.0]).T)
    c, slow = g.Context(0), g.Context(0)
    slow.set_tuning("set_select", 0)
    a, b = c.cloud(x, y, z), slow.cloud(x, y, z)
    k = min(8, n - 1)
    st = [g.stage(g.STAGE_COVFEAT, k, features=g.F_ALL10)]
    same_bits(b.run(st, init=np.nan), a.run(st, init=np.nan))
    assert np.array_equal(a.knn(k)[0], b.knn(k)[0])
    slow.close()
    c.close()


@pytest.mark.parametrize("n", [262080, 262144, 262209])
@pytest.mark.parametrize("kind", ["volume", "normal"])
def test_waves_searching_their_own_rows(kind, n):
    # The wave-per-query search beside the launch size from which its waves
    # search most of their uncertified rows themselves.
    rng = np.random.default_rng(n)
    p = rng.uniform(0, 50.0, (n, 3)) if kind == "volume" else rng.normal(size=(n, 3)) * [90, 90, 5]
    x, y, z = np.ascontiguousarray(p.T)
    c, slow = g.Context(0), g.Context(0)
    slow.set_tuning("set_select", 0)
    a, b = c.cloud(x, y, z), slow.cloud(x, y, z)
    st = [g.stage(g.STAGE_EIGENVALUES, 39)]
    same_bits(b.run(st, init=np.nan), a.run(st, init=np.nan))
    assert np.array_equal(a.knn(38)[0], b.knn(38)[0])
    slow.close()
    c.close()


def test_autotuner_tries_the_z_grouping(tmp_path):
    # From 38 entries on the z grouping shapes the search, and is tuned.
    c = g.Context(0)
    rng = np.random.default_rng(5)
    cl = c.cloud(*np.ascontiguousarray((rng.uniform(0, 40, (20000, 3)) * [1, 1, 0.1]).T))
    for knn, tuned in ((39, True), (16, False)):
        c.autotune(cl, [g.stage(g.STAGE_COVFEAT, knn)], factors=(0.6,))
        c.save_tuning(tmp_path / "t")
        rows = [r.split() for r in (tmp_path / "t").read_text().splitlines() if r[0] != "#"]
        assert any((int(r[3]) > 0) == tuned for r in rows), (knn, rows)
        if tuned:
            assert all(int(r[3]) > 0 for r in rows)
    c.close()


# 22 to 37 entries are searched by the query-per-lane search from 131,072
# points (of a cloud or batch) on: copies of a cloud side by side, beside that
# count, at the instance's limits.
@pytest.mark.parametrize("n", [131071, 131072, 131137])
@pytest.mark.parametrize("k", [22, 36, 37])
@pytest.mark.parametrize("kind", ["ragged", "clumps", "shells", "tower"])
def test_wide_neighborhoods_of_large_clouds(oracle, kind, k, n):
    p = np.array(path_cloud(kind)).T
    m = -(-n // len(p))
    p = np.concatenate([p + [5000.0 * i, 0.0, 0.0] for i in range(m)])[:n]
    x, y, z = np.ascontiguousarray(p.T)
    c, slow = g.Context(0), g.Context(0)
    slow.set_tuning("set_select", 0)
    cl = c.cloud(x, y, z)
    st = [g.stage(g.STAGE_COVFEAT, k - 1)]
    want = slow.cloud(x, y, z).run(st, init=np.nan)
    same_bits(cl.run(st, init=np.nan), want)
    if n == 131072:
        tree = oracle.kd3(x, y, z)
        assert set_equal_rows(cl.knn(k)[0], tree.neighbors_all(k, threads=8)).all()
    # The same points as a batch of two tiles.
    half = n // 2
    tiles = [(x[:half], y[:half], z[:half]), (x[half:], y[half:], z[half:])]
    b = c.batch(tiles)
    got = b.run(st, init=np.nan)
    for t in (0, 1):
        alone = slow.cloud(*tiles[t]).run(st, init=np.nan)
        same_bits(([[b.tile(col, t) for col in got[0][0]]], [b.tile(got[1][0], t)]), alone)
    b.close()
    slow.close()
    c.close()
