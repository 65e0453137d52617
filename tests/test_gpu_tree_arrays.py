"""Who owns the query-time arrays of photon trees that a caller made or batched: what is attached
can be released, and arrays that others may read are kept."""

import ctypes

import numpy as np
import pytest

from mnrt_amd import api, native as N
from helpers import f4

pytestmark = pytest.mark.gpu

LEAF = 3 << 30


def _caller_batch(cuda, refs):
    """A batch of single-leaf trees in the caller's own arrays; refs[s]: scene s's references."""
    elems = [max(r) + 1 for r in refs]
    off = np.concatenate([[0], np.cumsum(elems)]).astype(np.uint32)
    nodes = cuda.from_numpy(np.array([[len(r), LEAF] for r in refs], np.uint32).view(np.int32)).cuda()
    flat = cuda.from_numpy(np.concatenate(refs).astype(np.int32)).cuda()
    B = api.TreeBatch(N.KIND_POINT, off)
    first = 0
    for s, r in enumerate(refs):
        t = B.arr[s]
        t.kind, t.num_nodes, t.num_refs, t.num_elems, t.num_leaves = N.KIND_POINT, 1, len(r), elems[s], 1
        for a in range(3):
            t.root_min[a], t.root_max[a] = -1.0, 1.0
        t.d_nodes, t.d_refs = nodes.data_ptr() + 8 * s, flat.data_ptr() + 4 * first
        first += len(r)
    return B, [nodes, flat], int(off[-1])


def _photons(n, seed=0):
    rng = np.random.default_rng(seed)
    d = rng.normal(size=(n, 3))
    return f4(rng.uniform(-1, 1, (n, 3))), f4(rng.uniform(0, 1, (n, 3))), f4(d / np.linalg.norm(d, axis=1)[:, None])


def _release(tree):
    N.check(N.load().mnrt_tree_release(ctypes.byref(tree)), "mnrt_tree_release")


@pytest.mark.parametrize("refs", [
    [[0, 1, 2, 2, 1], [0, 1, 2, 3]],  # more references than elements: no hierarchies
    [[0, 1, 2], [1, 0, 3, 2]],        # hierarchies
])
def test_caller_batch_releases(cuda, refs):
    B, keep, n = _caller_batch(cuda, refs)
    ph = [api.dev(a) for a in _photons(n)]
    api.attach_photon_records_batch(B, *ph)
    boxes = all(len(r) == max(r) + 1 for r in refs)
    for s, r in enumerate(refs):
        assert bool(B.arr[s].owns_qnodes & N.QNODES_BOXES) == boxes
        q = ph[0][int(B.offsets[s]):int(B.offsets[s + 1])].contiguous()
        got = api.knn_radii(B[s], 2, 9.0, q).cpu().numpy()
        p = q.cpu().numpy()[:, :3]
        d = np.sort(np.linalg.norm(p[r][None] - p[:, None], axis=2), 1)[:, 1]
        assert np.allclose(got, d, rtol=1e-6, atol=1e-7)
    cuda.cuda.synchronize()
    _release(B.arr[0])
    assert not B.arr[0].d_recs and not B.arr[0].d_qnodes and B.arr[0].d_nodes
