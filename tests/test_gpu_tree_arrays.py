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


def _collapse(T, most):
    N.check(N.load().mnrt_tree_collapse(T.ref(), most, N.stream_handle()), "mnrt_tree_collapse")


def _radii(T, k, q):
    return api.knn_radii(T, k, 9.0, q).cpu().numpy()


def test_words_that_queries_read_are_kept(cuda):
    """Records in the caller's array, node words from mnrt_tree_collapse: queries can have read both
    when the records are attached again, so both stay where they are."""
    pos, power, pdir = (api.dev(a) for a in _photons(3000))
    want = api.build_points(pos)
    api.attach_photon_records(want, pos, power, pdir)
    T = api.build_points(pos)
    recs = cuda.empty(3000 * 8, dtype=cuda.float32, device="cuda")
    T.t.d_recs = recs.data_ptr()
    _collapse(T, 64)
    before = T.t.d_qnodes
    api.attach_photon_records(T, pos, power, pdir)
    assert T.t.d_qnodes == before and T.t.owns_qnodes == N.QNODES_OWNED
    assert np.array_equal(_radii(T, 20, pos[:500].contiguous()), _radii(want, 20, pos[:500].contiguous()))
    # without records before, no query can have: the words give way to a hierarchy with words
    U = api.build_points(pos)
    _collapse(U, 64)
    api.attach_photon_records(U, pos, power, pdir)
    assert U.t.owns_qnodes == N.QNODES_OWNED | N.QNODES_BOXES
    assert np.array_equal(_radii(U, 20, pos[:500].contiguous()), _radii(want, 20, pos[:500].contiguous()))
    for tree in (T, U, want):
        tree.release()


def test_first_tree_of_a_batch_keeps_the_shared_array(cuda):
    """Records attached again to the first tree of a batch without hierarchies, which owns the array
    that the other trees' node words lie in."""
    refs = [[0, 1, 2], [0, 1, 2, 2, 1]]
    B, keep, n = _caller_batch(cuda, refs)
    ph = [api.dev(a) for a in _photons(n)]
    api.attach_photon_records_batch(B, *ph)
    before = [B.arr[s].d_qnodes for s in range(2)]
    api.attach_photon_records(B[0], *(a[:3].contiguous() for a in ph))
    assert [B.arr[s].d_qnodes for s in range(2)] == before
    cuda.cuda.synchronize()
    _release(B.arr[0])
