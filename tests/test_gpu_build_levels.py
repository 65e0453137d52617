"""The level loop of the kd-tree build where its units change: nodes around a wave of 64
slots and around one pass of a node's wave counts (512 waves), single-element small roots, levels
that outgrow the first buffer sizes, and workgroups that span scenes.  Node words and references
equal the oracle's word for word."""

import numpy as np
import pytest

from mnrt_amd import api
from helpers import f4

pytestmark = pytest.mark.gpu


def _same(orc, kind, dt, v, small_max, root=None):
    ot = orc.build(kind, *v, small_max=small_max, root=root)
    assert np.array_equal(dt.nodes_host(), ot.nodes)
    assert np.array_equal(dt.refs_host(), ot.refs)
    assert np.array_equal(dt.root.view(np.uint32), ot.root.view(np.uint32))
    assert (dt.max_level, dt.t.num_leaves) == (ot.max_level, ot.num_leaves)


@pytest.mark.parametrize("n,small_max", [(2, 1), (3, 1), (200, 1), (33, 32), (64, 32), (65, 32), (65, 64), (127, 32),
                                         (128, 64), (129, 64), (4095, 32), (4097, 32), (32767, 32), (32768, 64),
                                         (32769, 32), (65537, 32), (200003, 17)])
@pytest.mark.parametrize("kind", [0, 1])
def test_level_units(orc, cuda, kind, n, small_max):
    rng = np.random.default_rng(n + kind)
    c = rng.uniform(-1.0, 1.0, (n, 3))
    c[: n // 3] = np.round(c[: n // 3] * 8) / 8  # planes shared by many elements, and split planes
    if kind == 0:
        v = [f4(c + rng.normal(scale=0.3 / np.cbrt(n), size=c.shape)) for _ in range(3)]
    else:
        v = [f4(c)]
    p = api.default_params(kind)
    p.small_node_max = small_max
    print(f"kind {kind} n {n} small_max {small_max}", flush=True)
    dt = api.build_tri(*v, p) if kind == 0 else api.build_points(v[0], p)
    cuda.cuda.synchronize()
    _same(orc, kind, dt, v, small_max)


@pytest.mark.parametrize("n,size,small_max", [(1200, 0.5, 8), (3000, 0.15, 2), (700, 1.0, 64)])
def test_levels_outgrow_first_buffers(orc, cuda, n, size, small_max):
    # triangles that straddle many splits: element copies, nodes and large-stage leaves beyond
    # what ordinary scenes need
    rng = np.random.default_rng(n)
    c = rng.uniform(-1.0, 1.0, (n, 3))
    v = [f4(c + rng.uniform(-size, size, c.shape)) for _ in range(3)]
    p = api.default_params(0)
    p.small_node_max = small_max
    print(f"overlapping: {n} triangles of {size}, small_max {small_max}", flush=True)
    dt = api.build_tri(*v, p)
    cuda.cuda.synchronize()
    _same(orc, 0, dt, v, small_max)


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("sizes", [[5000, 3, 4000, 0, 64, 65, 1, 9000, 100], [1] * 300 + [70] * 40 + [4096, 4096]])
def test_scenes_across_workgroups(orc, cuda, kind, sizes):
    rng = np.random.default_rng(len(sizes))
    off = np.zeros(len(sizes) + 1, np.uint32)
    off[1:] = np.cumsum(sizes)
    c = rng.uniform(-1.0, 1.0, (int(off[-1]), 3)) + np.repeat(rng.uniform(-9, 9, (len(sizes), 3)), sizes, axis=0)
    v = [f4(c + rng.normal(scale=0.02, size=c.shape)) for _ in range(3)] if kind == 0 else [f4(c)]
    print(f"kind {kind}: {len(sizes)} scenes", flush=True)
    B = api.build_tri_batch(*v, off) if kind == 0 else api.build_points_batch(v[0], off)
    cuda.cuda.synchronize()
    for s, n in enumerate(sizes):
        if n:
            _same(orc, kind, B[s], [a[off[s]:off[s + 1]] for a in v], 64 if kind == 0 else 32)
    B.release()
