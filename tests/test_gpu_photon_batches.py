"""Photon generation over several path batches: scenes where most paths are absorbed at once, where
few photons or none are stored at all, the fewest photons and bounces.  Photons, source paths and path
count equal the oracle's, which traces path by path."""

import numpy as np
import pytest

from mnrt_amd import api, scene as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("target,bounces,lit", [(1, 4, 1.0), (1, 0, 0.5), (300, 4, 0.02), (4097, 0, 1.0), (9001, 4, 0.1),
                                                (20000, 4, 0.3), (40000, 3, 0.6), (150, 4, 0.0)])
def test_batches(orc, cuda, target, bounces, lit):
    sc = S.scene_small(subdiv=3, num_lights=2)
    rng = np.random.default_rng(target)
    albedo = sc.albedo.copy()
    albedo[rng.random(len(albedo)) >= lit] = 0.0  # black: nothing is stored there
    eps = sc.ray_epsilon()
    T = api.build_tri(sc.v0, sc.v1, sc.v2)
    ot = orc.build(0, sc.v0, sc.v1, sc.v2)
    print(f"photons: target {target} bounces {bounces} lit {lit}", flush=True)
    g = api.photons_generate(T, sc.v0, sc.v1, sc.v2, albedo, sc.lights, target, bounces, 11, eps, want_meta=True)
    o = orc.photons(ot, sc.v0, sc.v1, sc.v2, albedo, sc.lights, target, bounces, 11, eps)
    cuda.cuda.synchronize()
    n = o["count"]
    assert (g["count"], g["paths"]) == (n, o["paths"])
    for key in ("pos", "power", "dir"):
        assert np.array_equal(g[key].cpu().numpy()[:n].view(np.uint32), o[key][:n].view(np.uint32)), key
    assert np.array_equal(g["path"].cpu().numpy()[:n].view(np.uint32), o["path"][:n])
