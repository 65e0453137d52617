"""Photon trees without a box hierarchy (node words that a caller supplies): radii, the adjoint and both
phases of a batch walk the node words and give what the hierarchy gives, bit for bit."""

import pytest
import torch

from mnrt_amd import api, native as N
from test_gpu_batch import _batch_io, _query_setup

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.contiguous().view(torch.int32)


def _words(tree):
    w = api.DeviceTree(N.KIND_POINT, N.Tree.from_buffer_copy(tree.t), batch=tree)  # a view: releases nothing
    w.t.owns_qnodes = 0
    return w


@pytest.mark.parametrize("k", [1, 50, 100, 256])
def test_words_equal_boxes(cuda, k):
    X = _query_setup(torch, [1500, 300, 4000], [6000, 200, 15000], [(40, 32), (8, 8), (48, 48)], seed=90)
    g = torch.Generator(device="cpu").manual_seed(k)
    n = int(X["roff"][-1])
    grad = (torch.rand((n, 4), generator=g) - 0.3).cuda()

    def run():
        Q = api.QueryBatch(X["TB"], X["toff"], X["roff"], X["eps"], X["PB"], X["rmax"], k)
        B = _batch_io(torch, Q, X, k)
        B["grad_rad4"] = grad
        B["out_count"] = torch.empty(n, dtype=torch.int32, device="cuda")
        B["grad_pow4"] = torch.zeros((int(Q.photon_offsets[-1]), 4), device="cuda")
        B["grad_clr4"] = torch.zeros((n, 4), device="cuda")
        B["out_nbr"].zero_()
        B["out_r2"].zero_()
        B["out_count"].zero_()
        Q.make_io(**B)
        Q.run(7)
        Q.run(8)
        torch.cuda.synchronize()
        Q.close()
        return B

    print(f"k {k}: batch over hierarchies", flush=True)
    boxes = run()
    owned = [t.owns_qnodes for t in X["PB"].arr]
    assert all(o & N.QNODES_BOXES for o in owned)
    for t in X["PB"].arr:
        t.owns_qnodes = 0
    try:
        print("batch over node words", flush=True)
        words = run()
    finally:
        for t, o in zip(X["PB"].arr, owned):
            t.owns_qnodes = o
    for c in ("io_rad4", "out_r2", "out_nbr", "out_count", "grad_pow4", "grad_clr4"):
        assert torch.equal(_bits(boxes[c]), _bits(words[c])), c
    cnt = boxes["sp_count"].cpu().numpy()
    for s in range(3):
        a, m, tree, r = int(X["roff"][s]), int(cnt[s]), X["PB"][s], float(X["rmax"][s])
        q = [boxes[c][a:a + m].contiguous() for c in ("sp_pos4", "sp_nrm4", "sp_dir4", "sp_infl4", "sp_clr4")]
        print(f"scene {s}: radii and adjoint", flush=True)
        assert torch.equal(_bits(api.knn_radii(tree, k, r, q[0])), _bits(api.knn_radii(_words(tree), k, r, q[0])))
        rest = [grad[a:a + m], boxes["out_r2"][a:a + m].contiguous(), boxes["out_count"][a:a + m].contiguous()]
        one, two = (api.knn_gather_bwd(t, k, r, *q, *rest) for t in (tree, _words(tree)))
        for x, y in zip(one, two):
            assert torch.equal(_bits(x), _bits(y))
        p0 = int(X["poff"][s])
        assert torch.equal(_bits(two[0]), _bits(words["grad_pow4"][p0:int(X["poff"][s + 1])]))
