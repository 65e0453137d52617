"""Host-driven builds that outgrow their first buffers, at one level or at many, and go on from there:
single trees and batches.  Node words and references equal the oracle's word for word, and a
recorded build made from such a build replays to the same trees."""

import numpy as np
import pytest

from mnrt_amd import api, native as N
from helpers import f4

pytestmark = pytest.mark.gpu


def _same(orc, kind, dt, v, small_max):
    ot = orc.build(kind, *v, small_max=small_max)
    assert np.array_equal(dt.nodes_host(), ot.nodes)
    assert np.array_equal(dt.refs_host(), ot.refs)
    assert (dt.max_level, dt.t.num_leaves) == (ot.max_level, ot.num_leaves)


def _tris(rng, n, size):
    c = rng.uniform(-1.0, 1.0, (n, 3))
    return [f4(c + rng.uniform(-size, size, c.shape)) for _ in range(3)]


@pytest.mark.parametrize("n,size,small_max", [(900, 0.3, 1), (3000, 0.1, 1), (3000, 0.1, 4), (20000, 0.01, 2),
                                              (2000, 0.5, 16), (65, 2.0, 1)])
def test_triangles(orc, cuda, n, size, small_max):
    v = _tris(np.random.default_rng(n), n, size)
    p = api.default_params(0)
    p.small_node_max = small_max
    print(f"{n} triangles of {size}, small_max {small_max}", flush=True)
    for _ in range(2):  # the workspace of the first is there for the second
        dt = api.build_tri(*v, p)
        cuda.cuda.synchronize()
        _same(orc, 0, dt, v, small_max)
        dt.release()


@pytest.mark.parametrize("n,cells,small_max", [(20000, 4, 32), (30000, 8, 1), (5000, 1, 8)])
def test_points_in_few_places(orc, cuda, n, cells, small_max):
    # more points in a place than a small root holds: those nodes are split to the last level
    v = [f4(np.round(np.random.default_rng(n).uniform(0, cells, (n, 3))) / cells)]
    p = api.default_params(1)
    p.small_node_max = small_max
    print(f"{n} points in {(cells + 1) ** 3} places, small_max {small_max}", flush=True)
    dt = api.build_points(v[0], p)
    cuda.cuda.synchronize()
    _same(orc, 1, dt, v, small_max)


def test_batch_and_recorded_build(orc, cuda):
    rng = np.random.default_rng(7)
    sizes, small_max = [700, 40, 1500, 0, 3, 900], 2
    off = np.zeros(len(sizes) + 1, np.uint32)
    off[1:] = np.cumsum(sizes)
    v = [np.concatenate(a) for a in zip(*[_tris(rng, n, 0.4) for n in sizes])]
    p = api.default_params(0)
    p.small_node_max = small_max
    print("batch", flush=True)
    B = api.build_tri_batch(*v, off, p)
    print("recorded", flush=True)
    G = api.BuildGraph(N.KIND_TRI, off, *v, params=p)
    for _ in range(2):
        G.replay()
        assert G.status() == 0
    for s, n in enumerate(sizes):
        if n:
            _same(orc, 0, B[s], [a[off[s]:off[s + 1]] for a in v], small_max)
            assert np.array_equal(G.trees[s].nodes_host(), B[s].nodes_host())
            assert np.array_equal(G.trees[s].refs_host(), B[s].refs_host())
    G.close()
    B.release()
