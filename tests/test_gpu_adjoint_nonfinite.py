"""The kNN adjoint of gradients that are not finite: one NaN or infinite channel of one query
makes the photon gradients of its map NaN (a fixed-point sum has no such value), in the single
call and per scene of a batch; the other queries' colour gradients and the other scenes are the
bits they are without it."""

import pytest

from mnrt_amd import api
from test_gpu_batch import _batch_io, _query_setup

pytestmark = pytest.mark.gpu

K = 50


def _setup(torch):
    X = _query_setup(torch, [1500, 900], [6000, 4000], [(40, 32), (24, 24)], seed=90)
    Q = api.QueryBatch(X["TB"], X["toff"], X["roff"], X["eps"], X["PB"], X["rmax"], K)
    B = _batch_io(torch, Q, X, K)
    n = int(X["roff"][-1])
    B["grad_rad4"] = torch.rand((n, 4), generator=torch.Generator(device="cpu").manual_seed(1)).cuda() - 0.3
    B["out_count"] = torch.empty(n, dtype=torch.int32, device="cuda")
    B["grad_pow4"] = torch.zeros((int(Q.photon_offsets[-1]), 4), device="cuda")
    B["grad_clr4"] = torch.zeros((n, 4), device="cuda")
    Q.make_io(**B)
    Q.run(7)
    return X, Q, B


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("channel", [0, 1, 2])
def test_not_finite(cuda, value, channel):
    torch = cuda
    X, Q, B = _setup(torch)
    m, P0 = int(B["sp_count"][0]), int(Q.photon_offsets[1])
    at = int(torch.nonzero(B["out_count"][:m] >= K)[7])
    grad = B["grad_rad4"].clone()

    def batch():
        Q.run(8)
        return B["grad_pow4"].clone(), B["grad_clr4"].clone()

    def single():
        return api.knn_gather_bwd(X["PB"][0], K, float(X["rmax"][0]),
                                  *(B[c][:m].contiguous() for c in ("sp_pos4", "sp_nrm4", "sp_dir4", "sp_infl4",
                                                                    "sp_clr4", "grad_rad4", "out_r2", "out_count")))

    clean, clean1 = batch(), single()
    assert torch.isfinite(clean[0]).all() and torch.isfinite(clean1[0]).all()
    B["grad_rad4"][at, channel] = value
    bad, bad1 = batch(), single()
    others = torch.arange(m, device="cuda") != at
    for gp in (bad[0][:P0], bad1[0]):
        assert torch.isnan(gp[:, :3]).all() and (gp[:, 3] == 0).all()
    assert torch.equal(bad[0][P0:].view(torch.int32), clean[0][P0:].view(torch.int32))
    assert torch.equal(bad[1][:m][others].view(torch.int32), clean[1][:m][others].view(torch.int32))
    assert torch.equal(bad1[1][others].view(torch.int32), clean1[1][others].view(torch.int32))
    assert not torch.isfinite(bad1[1][at, channel])
    # and back
    B["grad_rad4"].copy_(grad)
    again, again1 = batch(), single()
    assert torch.equal(again[0].view(torch.int32), clean[0].view(torch.int32))
    assert torch.equal(again1[0].view(torch.int32), clean1[0].view(torch.int32))
    Q.close()
