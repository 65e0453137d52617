"""Launches of more windows of rays than waves that run at once, where a wave whose rays do not go
together takes windows from the launch's end: every ray is traced, whatever mix of rays the windows
hold, and two launches on two streams do not meet.  Compared with the same rays in launches of a
wave per window, which the oracle covers."""

import numpy as np
import pytest

from mnrt_amd import api, scene as S

pytestmark = pytest.mark.gpu

WINDOWS = 9216 * 64  # rays up to which every window has its own wave


@pytest.fixture(scope="module")
def tree(cuda):
    sc = S.scene_small(subdiv=3)
    return api.build_tri(sc.v0, sc.v1, sc.v2)


def _rays(torch, n, kind, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    o = torch.rand((n, 4), device="cuda", generator=g) * 1.8 - 0.9
    d = torch.randn((n, 4), device="cuda", generator=g)
    i = torch.arange(n, device="cuda")
    if kind != "random":
        together = (i * 3 // n == 0) if kind == "mixed" else torch.zeros(n, dtype=torch.bool, device="cuda")
        miss = (i * 3 // n == 1) if kind == "mixed" else torch.ones(n, dtype=torch.bool, device="cuda")
        if kind == "alternating":
            together, miss = (i // 64) % 3 == 0, (i // 64) % 3 == 1
        w = 1200
        cam = torch.stack([(i % w) / w - 0.5, ((i // w) % w) / w - 0.5, torch.full((n,), -1.0, device="cuda"),
                           torch.zeros(n, device="cuda")], 1)
        d = torch.where(together[:, None], cam, d)
        o = torch.where(together[:, None], torch.tensor([0.0, 0.0, 0.9, 0.0], device="cuda"), o)
        o = torch.where(miss[:, None], torch.tensor([0.0, 0.0, 3.0, 0.0], device="cuda"), o)
        d = torch.where(miss[:, None], torch.tensor([0.0, 0.1, 1.0, 0.0], device="cuda"), d)
    return o.contiguous(), d.contiguous()


def _pieces(torch, tree, o, d):
    out = [api.trace_closest(tree, o[a:a + 400000].contiguous(), d[a:a + 400000].contiguous(), 1e-4, want_pt=True)
           for a in range(0, len(o), 400000)]
    return [torch.cat([p[c] for p in out]) for c in range(4)]


def _same(torch, a, b):
    for x, y in zip(a, b):
        assert torch.equal(x.view(torch.int32), y.view(torch.int32))


@pytest.mark.parametrize("n", [WINDOWS, WINDOWS + 1, WINDOWS + 64, 1000003, 2073600])
@pytest.mark.parametrize("kind", ["random", "mixed", "alternating", "miss"])
def test_every_ray(cuda, tree, n, kind):
    print(f"{n} rays, {kind}", flush=True)
    o, d = _rays(cuda, n, kind, n)
    got = api.trace_closest(tree, o, d, 1e-4, want_pt=True)
    want = _pieces(cuda, tree, o, d)
    _same(cuda, got, want)
    if kind == "miss":
        assert (got[0] == -1).all()
    else:
        assert (got[0] >= 0).sum() > n // 4


def test_two_streams(cuda, tree):
    torch = cuda
    rays = [_rays(torch, 700003 + 1000 * s, k, s) for s, k in enumerate(("random", "alternating"))]
    want = [_pieces(torch, tree, *r) for r in rays]
    streams = [torch.cuda.Stream() for _ in rays]
    torch.cuda.synchronize()
    got = []
    for s, r in zip(streams, rays):
        with torch.cuda.stream(s):
            got.append([api.trace_closest(tree, *r, 1e-4, want_pt=True) for _ in range(3)])
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        for one in g:
            _same(torch, one, w)
