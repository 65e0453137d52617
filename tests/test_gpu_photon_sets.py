"""Photon tracing with 32 and 64 paths a wave at once: paths refill and share tests from the first ray
on, never walking as one set.  Photons equal the oracle's bit for bit."""

import numpy as np
import pytest

from mnrt_amd import api, scene as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("target,bounces", [(330000, 4), (660000, 4), (140001, 0)])
def test_wide_sets(orc, cuda, target, bounces):
    sc = S.scene_small(subdiv=2)
    eps = sc.ray_epsilon()
    T = api.build_tri(sc.v0, sc.v1, sc.v2)
    print(f"{target} photons, {bounces} bounces", flush=True)
    got = api.photons_generate(T, sc.v0, sc.v1, sc.v2, sc.albedo, sc.lights, target, bounces, 7, eps)
    want = orc.photons(orc.build(0, sc.v0, sc.v1, sc.v2), sc.v0, sc.v1, sc.v2, sc.albedo, sc.lights, target, bounces, 7,
                       eps)
    assert got["count"] == want["count"] == target and got["paths"] == want["paths"]
    for c in ("pos", "power", "dir"):
        assert np.array_equal(got[c].cpu().numpy().view(np.uint32), want[c].view(np.uint32)), c
