"""The search's kernel instances and its paths for crowded and sparse rows:
lists hold the oracle's KD3 neighbors and feature columns and statuses equal the
growing search's, bit for bit, at the capacities where the instance changes
and at row counts beside multiples of the wave's 64 queries."""
import numpy as np
import pytest

import gpupdal_amd as g
from helpers import set_equal_rows, small_cloud

pytestmark = pytest.mark.gpu


@pytest.fixture
def ctx():
    # One of this test's own: the flags of re-solved rows follow the grid, and
    # a shared context may hold autotuned grids.
    c = g.Context(0)
    yield c
    c.close()


def cloud(kind):
    rng = np.random.default_rng(81)
    if kind == "ragged":  # last wave of one query
        x, y, z = small_cloud(4097, seed=82, dup_frac=0.01)
    elif kind == "few":  # fewer queries than a wave
        x, y, z = small_cloud(61, seed=83)
    elif kind == "clumps":  # a sparse surface with dense balls: crowded boxes
        c = rng.uniform(0, 300.0, (6, 3)) * [1, 1, 0.05]
        p = np.concatenate([rng.uniform(0, 300.0, (3000, 3)) * [1, 1, 0.02]] +
                           [q + rng.normal(0, 0.4, (900, 3)) for q in c])
        x, y, z = np.ascontiguousarray(p.T)
    elif kind == "shells":  # spacing over four decades, far from the origin
        r = 10.0 ** rng.uniform(-2, 2, 6000)
        u = rng.normal(size=(6000, 3))
        p = r[:, None] * u / np.linalg.norm(u, axis=1)[:, None] + [5e5, 4e6, 100.0]
        x, y, z = np.ascontiguousarray(p.T)
    else:  # "tower": coincident points and one tall column
        p = np.concatenate([np.repeat(rng.uniform(0, 20.0, (60, 3)), 40, axis=0),
                            np.column_stack([np.full(1700, 5.0), np.full(1700, 5.0),
                                             rng.uniform(0, 900.0, 1700)])])
        x, y, z = np.ascontiguousarray(p.T)
    return x, y, z


# Result capacities beside each change of instance: k for lists; features
# search for one entry more.
@pytest.mark.parametrize("k", [1, 8, 9, 10, 20, 21, 22, 36, 37, 38, 62])
@pytest.mark.parametrize("kind", ["ragged", "few", "clumps", "shells", "tower"])
def test_paths_agree(ctx, oracle, kind, k):
    if kind == "few" and k > 36:
        pytest.skip("fewer points than neighbors is covered elsewhere")
    x, y, z = cloud(kind)
    cl = ctx.cloud(x, y, z)
    ids, _ = cl.knn(k)
    tree = oracle.kd3(x, y, z)
    assert set_equal_rows(ids, tree.neighbors_all(k, threads=8)).all(), "lists"
    sts = [[g.stage(g.STAGE_COVFEAT, k, features=g.F_ALL10)]]
    if 2 * k <= 62:
        sts.append([g.stage(g.STAGE_COVFEAT, k, stride=2)])
    slow = g.Context(0)
    slow.set_tuning("set_select", 0)
    cs = slow.cloud(x, y, z)
    for st in sts:
        a, b = cl.run(st, init=np.nan), cs.run(st, init=np.nan)
        assert np.array_equal(a[1][0], b[1][0]), st[0].stride
        for ca, cb in zip(a[0][0], b[0][0]):
            assert np.array_equal(np.asarray(ca).view(np.uint64), np.asarray(cb).view(np.uint64))
    cs.close()
    slow.close()


@pytest.mark.parametrize("knns", [[8, 16, 32], [8, 40], [62], [21, 9, 36, 37, 50]])
def test_batch_instances_agree(knns):
    # Tiles served by different instances share a batch: each tile's columns
    # are those of the tile run alone.
    out = {}
    tiles = [small_cloud(1500 + 64 * i + i, seed=90 + i) for i in range(len(knns))]
    with_k = [g.stage(g.STAGE_COVFEAT, 8)]
    c = g.Context(0)
    b = c.batch(tiles)
    out["batch"] = b.run(with_k, tile_knn=knns, init=np.nan)
    for t, (xyz, k) in enumerate(zip(tiles, knns)):
        one = c.cloud(*xyz).run([g.stage(g.STAGE_COVFEAT, k)], init=np.nan)
        for ca, cb in zip(one[0][0], out["batch"][0][0]):
            assert np.array_equal(np.asarray(ca).view(np.uint64),
                                  np.asarray(b.tile(cb, t)).view(np.uint64)), (t, k)
    b.close()
    c.close()


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 4097])
@pytest.mark.parametrize("per", [4, 40, 250, 450, 900])
def test_radius_paths_agree(ctx, oracle, n, per):
    # From a few neighbors (whole groups staged) over halved groups to rows
    # streamed one by one, and waves with both.  Counts are exact; moments of
    # up to n points of size r differ from numpy's by n eps r^2.
    rng = np.random.default_rng(84)
    p = np.column_stack([rng.uniform(0, 40.0, (n, 2)), rng.uniform(0, 0.4, n)])
    p[n // 2:, :2] *= 0.25
    r = float(np.sqrt(per * 1600.0 / (np.pi * n)))
    x, y, z = np.ascontiguousarray(p.T)
    cl = ctx.cloud(x, y, z)
    want = oracle.kd3(x, y, z).radius_counts(r)
    assert np.array_equal(cl.radius_counts(r), want)
    (cols,), (status,) = cl.run([g.stage(g.STAGE_EIGENVALUES, 8, radius=r, min_k=3)],
                                init=np.nan)
    cl.close()
    rows = np.flatnonzero(want >= 3)[::37]
    got = np.array([c[rows] for c in cols]).T
    d = p[rows][:, None, :] - p[None]
    near = np.einsum("ijk,ijk->ij", d, d) < r * r
    for i, m in zip(range(len(rows)), near):
        if m.sum() != want[rows[i]]:
            continue  # a distance that rounds to r otherwise than KD3Index's
        ev = np.linalg.eigvalsh(np.cov(p[m].T))
        tol = 64 * m.sum() * np.finfo(np.float64).eps * max(r * r, ev[-1])
        assert np.all(np.abs(got[i] - ev) <= tol), (n, per, rows[i])
