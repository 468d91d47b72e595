"""The exact tree's middle nodes (split by one workgroup each): the tree equals
the oracle's KD3 tree, node for node, at point counts beside the limits of the
regimes and on clouds whose midpoint cuts make long chains of uneven nodes."""
import numpy as np
import pytest

import gpupdal_amd as g
import oracle_lib as ol
from test_gpu_parity import _oracle_nodes, _tree_nodes

pytestmark = pytest.mark.gpu


def cloud(kind, n):
    rng = np.random.default_rng(n)
    if kind == "even":
        p = rng.uniform(0, 100.0, (n, 3))
    elif kind == "chain":  # halving the box takes off a few points at a time
        p = 10.0 ** rng.uniform(-6, 3, (n, 1)) * rng.uniform(0.5, 1.0, (n, 3))
    elif kind == "lattice":  # most cuts fall on points: second passes move them
        p = np.floor(rng.uniform(0, 12.0, (n, 3))) * 0.5
    else:  # "point": every point at one of two places
        p = np.where(rng.uniform(size=(n, 1)) < 0.3, 1.0, 2.0) * np.ones((n, 3))
    return np.ascontiguousarray(p.T)


@pytest.mark.parametrize("kind", ["even", "chain", "lattice", "point"])
@pytest.mark.parametrize("n,sub", [(2048, 2048), (2049, 2048), (4097, 4096), (32768, 2048),
                                   (32769, 2048), (70000, 2048), (1700, 101), (1616, 101),
                                   (9000, 512)])
def test_middle_nodes_equal_kd3(kind, n, sub):
    x, y, z = cloud(kind, n)
    c = g.Context(0)
    c.set_tuning("kd_subtree", sub)
    t = c.cloud(x, y, z).kdtree()
    c.close()
    e = ol.Oracle().kd3(x, y, z).export()
    assert np.array_equal(t["vind"].astype(np.uint64), e["vind"])
    assert _tree_nodes(t) == _oracle_nodes(e)
