"""Batched traces around the sizes where a wave's unit changes: sets of 16, 32 and 64 rays, and four
sets of 64 in batches of more than 6.3M rays, with scenes that end inside a unit.  Hits equal
those of the single-scene trace bit for bit."""

import numpy as np
import pytest

from mnrt_amd import api, native as N, scene as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rays", [[1, 15, 1000], [98304, 1, 0], [98305, 7], [150000, 46609], [200001, 193217],
                                  [3200001, 5, 3091454], [3200001, 5, 3091449]])
def test_units(cuda, rays):
    torch = cuda
    scs = [S.scene_sized(300 + 400 * i, seed=i) for i in range(len(rays))]
    trees = [api.build_tri(s.v0, s.v1, s.v2) for s in scs]
    toff, roff = np.zeros(len(rays) + 1, np.uint32), np.zeros(len(rays) + 1, np.uint32)
    toff[1:], roff[1:] = np.cumsum([s.num_tris for s in scs]), np.cumsum(rays)
    eps = np.array([s.ray_epsilon() for s in scs], np.float32)
    n = int(roff[-1])
    print(f"{n} rays in {len(rays)} scenes", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    o = torch.rand((n, 4), device="cuda", generator=g) * 1.8 - 0.9
    d = torch.randn((n, 4), device="cuda", generator=g)
    Q = api.QueryBatch(trees, toff, roff, eps)
    b = dict(orig4=o, dir4=d, hit_tri=torch.full((n,), -2, dtype=torch.int32, device="cuda"),
             hit_t=torch.empty(n, device="cuda"))
    Q.make_io(**b)
    Q.run(N.PHASE_TRACE)
    torch.cuda.synchronize()
    for s, t in enumerate(trees):
        a, e = int(roff[s]), int(roff[s + 1])
        if a == e:
            continue
        tri, lam, _, _ = api.trace_closest(t, o[a:e].contiguous(), d[a:e].contiguous(), float(eps[s]))
        assert torch.equal(b["hit_tri"][a:e], tri), s
        assert torch.equal(b["hit_t"][a:e].view(torch.int32), lam.view(torch.int32)), s
    Q.close()
