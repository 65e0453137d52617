"""kNN launches whose waves answer chains of queries: each starts from the one before it, and the
candidate buffer fills within a search.  Sets equal the brute force, sums the walk over the
query-time node words."""

import numpy as np
import pytest

from mnrt_amd import api, native as N
from helpers import f4

pytestmark = pytest.mark.gpu

ROOT = np.array([-1, -1, -1, 1, 1, 1], np.float32)


def _map(rng, n):
    # a thin volume, a dense spot and a grid with ties
    a = rng.uniform(-1, 1, (n, 3))
    a[: n // 2] = 0.3 + rng.normal(scale=0.01, size=(n // 2, 3))
    a[n // 2: n // 2 + n // 8] = np.round(a[n // 2: n // 2 + n // 8] * 10) / 10
    d = rng.normal(size=(n, 3))
    return f4(a.clip(-1, 1)), f4(rng.uniform(0, 1, (n, 3))), f4(d / np.linalg.norm(d, axis=1, keepdims=True))


def _path(rng, n):
    # small steps through the dense spot and out of it, with jumps between
    step = rng.normal(scale=0.004, size=(n, 3))
    q = np.cumsum(step, 0)
    q = q - q[(np.arange(n) // 512) * 512] + rng.uniform(-0.9, 0.9, (n // 512 + 1, 3))[np.arange(n) // 512]
    q[np.arange(n) // 512 % 2 == 0] = 0.3 + (q[np.arange(n) // 512 % 2 == 0] - 0.3) * 0.05
    return q.clip(-1.2, 1.2)


@pytest.mark.parametrize("k,rmax", [(1, 0.3), (50, 2.0), (50, 0.05), (256, 0.5)])
@pytest.mark.parametrize("order", ["path", "shuffled"])
def test_chains(orc, cuda, order, k, rmax):
    rng = np.random.default_rng(k)
    pos, power, pdir = _map(rng, 6000)
    n = 50021  # chains of two, the last of one
    qp = _path(rng, n)
    if order == "shuffled":
        qp = qp[rng.permutation(n)]
    nrm = rng.normal(size=(n, 3))
    q = dict(pos=f4(qp), nrm=f4(nrm), dir=f4(-nrm), infl=f4(np.ones((n, 3))), clr=np.ones((n, 4), np.float32))
    P = api.build_points(pos, api.default_params(N.KIND_POINT, ROOT, rmax))
    api.attach_photon_records(P, pos, power, pdir)
    words = api.DeviceTree(N.KIND_POINT, N.Tree.from_buffer_copy(P.t), batch=P)  # a view: releases nothing
    words.t.owns_qnodes = 0
    print(f"{n} queries, {order}, k {k}, radius {rmax}", flush=True)
    got = {}
    for name, tree in (("boxes", P), ("words", words)):
        out = api.knn_gather(tree, k, rmax, *(q[c] for c in ("pos", "nrm", "dir", "infl", "clr")), want_nbr=True,
                             want_r2=True, want_count=True)
        got[name] = {c: out[c].cpu().numpy().view(np.uint32) for c in ("rad", "nbr", "r2", "count")}
    nbr, cnt = orc.knn_brute(pos, q["pos"], k, rmax)
    for name, g in got.items():
        assert np.array_equal(g["count"], cnt), name
        assert np.array_equal(g["nbr"], nbr), name
    for c in ("rad", "r2"):
        assert np.array_equal(got["boxes"][c], got["words"][c]), c


@pytest.mark.parametrize("n,rmax", [(12 * 8192 * 16 - 1, 0.4), (12 * 8192 * 16, 0.4), (8 * 24576 + 5, 0.4),
                                    (8 * 24576 + 5, 0.03), (12 * 8192 * 16, 0.03)])
def test_long_chains(orc, cuda, n, rmax):
    # chains of 8, and of 16 from a dozen rounds of waves on; over node words 8 at most.  Within the small
    # radius most queries find fewer than k, one after the other, and some find more
    rng = np.random.default_rng(n)
    pos, power, pdir = _map(rng, 4000)
    qp = f4(_path(rng, n))
    q = [api.dev(a) for a in (qp, f4(np.ones((n, 3))), f4(-np.ones((n, 3))), f4(np.ones((n, 3))))]
    P = api.build_points(pos, api.default_params(N.KIND_POINT, ROOT, rmax))
    api.attach_photon_records(P, pos, power, pdir)
    words = api.DeviceTree(N.KIND_POINT, N.Tree.from_buffer_copy(P.t), batch=P)
    words.t.owns_qnodes = 0
    print(f"{n} queries, radius {rmax}", flush=True)
    a, b = (api.knn_gather(t, 10, rmax, *q, want_nbr=True, want_r2=True, want_count=True) for t in (P, words))
    for c in ("rad", "nbr", "r2", "count"):
        assert cuda.equal(a[c].view(cuda.int32), b[c].view(cuda.int32)), c
    some = np.concatenate([np.arange(2000), rng.integers(0, n, 2000), np.arange(n - 2000, n)])
    nbr, cnt = orc.knn_brute(pos, qp[some], 10, rmax)
    assert np.array_equal(a["count"].cpu().numpy().view(np.uint32)[some], cnt)
    assert np.array_equal(a["nbr"].cpu().numpy().view(np.uint32)[some], nbr)
    found = a["count"].cpu().numpy()
    assert (found >= 10).any() and ((found < 10).mean() > 0.2) == (rmax < 0.1)
