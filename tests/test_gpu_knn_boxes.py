"""kNN through the box hierarchy of a photon tree (mnrt_tree_attach_photon_records) at the
sizes where its levels begin and end, against the brute force and against the walk over the
query-time node words, which trees with caller-supplied words take."""

import numpy as np
import pytest

from mnrt_amd import api, native as N
from helpers import f4

pytestmark = pytest.mark.gpu

ROOT = np.array([-1, -1, -1, 1, 1, 1], np.float32)


def _inputs(n, rng):
    # a coarse grid of positions: many exact ties; equal powers whose sums need every bit
    pos = f4(np.round(rng.uniform(-1, 1, (n, 3)) * 40) / 40)
    power = f4(np.where(rng.uniform(size=(n, 1)) < 0.5, 1.0 + 2.0 ** -16, rng.uniform(0, 1, (n, 3))))
    d = rng.normal(size=(n, 3))
    pdir = f4(d / np.linalg.norm(d, axis=1, keepdims=True))
    qp = np.concatenate([rng.uniform(-1, 1, (120, 3)), pos[rng.integers(0, n, 60), :3],
                         rng.uniform(-9, 9, (20, 3)), [[np.nan, 0, 0], [0, 0, np.nan]]])
    m = len(qp)
    nrm = np.eye(3)[rng.integers(0, 3, m)]
    nrm[::3] = rng.normal(size=(m, 3))[::3]
    q = dict(pos=f4(qp), nrm=f4(nrm), dir=f4(rng.normal(size=(m, 3))), infl=f4(np.ones((m, 3))),
             clr=np.concatenate([rng.uniform(0, 1, (m, 3)), np.ones((m, 1))], 1).astype(np.float32))
    return pos, power, pdir, q


def _gather(tree, k, rmax, q, **more):
    out = api.knn_gather(tree, k, rmax, *(q[c] for c in ("pos", "nrm", "dir", "infl", "clr")), want_r2=True,
                         want_count=True, **more)
    return {c: t.cpu().numpy().view(np.uint32) for c, t in out.items() if t is not None}


@pytest.mark.parametrize("k,rmax", [(1, 0.4), (50, 0.4), (100, 1e30), (256, 0.4)])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 4095, 4096, 4097, 262145])
def test_boxes_equal_brute_force_and_node_words(orc, cuda, n, k, rmax):
    pos, power, pdir, q = _inputs(n, np.random.default_rng(n + k))
    P = api.build_points(pos, api.default_params(N.KIND_POINT, ROOT, 0.4))
    api.attach_photon_records(P, pos, power, pdir)
    assert P.t.owns_qnodes == N.QNODES_OWNED | N.QNODES_BOXES
    boxes = _gather(P, k, rmax, q, want_nbr=True)
    free = _gather(P, k, rmax, q)
    words = api.DeviceTree(N.KIND_POINT, N.Tree.from_buffer_copy(P.t), batch=P)  # a view: releases nothing
    words.t.owns_qnodes = 0
    walk = _gather(words, k, rmax, q, want_nbr=True)
    for c in boxes:
        assert np.array_equal(boxes[c], walk[c]), c
        assert c == "nbr" or np.array_equal(boxes[c], free[c]), c
    real = slice(0, len(q["pos"]) - 2)  # the last two queries have a NaN coordinate: no neighbours
    assert (boxes["count"][-2:] == 0).all() and (boxes["nbr"][-2:] == 0xFFFFFFFF).all()
    nbr, cnt = orc.knn_brute(pos, q["pos"][real], k, rmax)
    assert np.array_equal(boxes["count"][real], cnt) and np.array_equal(boxes["nbr"][real], nbr)
    o32 = orc.radiance(nbr, cnt, k, rmax, pos, power, pdir, *(q[c][real] for c in ("pos", "nrm", "dir", "infl", "clr")))[0]
    assert np.array_equal(boxes["rad"][real], o32.view(np.uint32))
