"""Ray launches at the sizes where a wave's share changes: fewer rays than lanes, the widths of 16,
32 and 64 rays a wave, partial windows, and waves that take further windows from a counter; with rays that
miss, leaves of very different sizes and equal lambdas.  Closest hits (index, lambda, barycentrics)
and occlusion equal the oracle's bit for bit."""

import numpy as np
import pytest

from mnrt_amd import api, scene as S
from helpers import f4

pytestmark = pytest.mark.gpu


def _scene():
    # scattered triangles and a stack of 70 equal ones (a leaf fuller than a wave, all lambdas equal)
    rng = np.random.default_rng(31)
    c = rng.uniform(-1.0, 1.0, (900, 1, 3)) * [1.0, 1.0, 0.3]
    t = c + rng.normal(scale=0.12, size=(900, 3, 3))
    same = np.repeat(np.array([[[-0.4, -0.4, 0.5], [0.4, -0.4, 0.5], [0.0, 0.5, 0.5]]]), 70, axis=0)
    t = np.concatenate([t[:450], same, t[450:]]).astype(np.float32)
    return [f4(t[:, k]) for k in range(3)]


@pytest.fixture(scope="module")
def trees(orc, cuda):
    v = _scene()
    T = orc.build(0, *v)
    DT = api.tree_from_host(0, T.nodes, T.refs, T.root, len(v[0]), T.max_level)
    api.attach_tri_records(DT, *v)
    return v, T, DT


@pytest.mark.parametrize("n", [1, 15, 16, 17, 1000, 32767, 32768, 32769, 65535, 65536, 65537, 98305, 196609, 589824, 589825, 700001])
def test_ray_counts(orc, cuda, trees, n):
    v, T, DT = trees
    rng = np.random.default_rng(n)
    o = f4(rng.uniform(-1.6, 1.6, (n, 3)))  # some outside the root box
    d = rng.normal(size=(n, 3))
    d[rng.random(n) < 0.1] *= [0.0, 0.0, 1.0]  # along an axis
    d[np.linalg.norm(d, axis=1) == 0.0] = [0.0, 1.0, 0.0]
    d = f4(d / np.linalg.norm(d, axis=1, keepdims=True))
    eps = 1e-4
    print(f"{n} rays", flush=True)
    tri, t, uv, _ = orc.trace(T, *v, o, d, eps)
    gtri, gt, guv, _ = [x.cpu().numpy() if x is not None else None for x in api.trace_closest(DT, o, d, eps)]
    assert np.array_equal(gtri, tri), f"{(gtri != tri).sum()} hit indices differ"
    assert np.array_equal(gt.view(np.uint32), t.view(np.uint32))
    assert np.array_equal(guv.view(np.uint32), uv.view(np.uint32))
    tmax = rng.uniform(0.0, 2.0, size=n).astype(np.float32)
    h, _ = orc.trace_any(T, T.root, *v, o, d, eps, tmax)
    assert np.array_equal(api.trace_any(DT, o, d, eps, tmax).cpu().numpy().astype(np.uint32), h)


def test_odd_rays_leave_the_others_alone(orc, cuda, trees):
    v, T, DT = trees
    rng = np.random.default_rng(3)
    n = 3000
    o, d = f4(rng.uniform(-1.0, 1.0, (n, 3))), f4(rng.normal(size=(n, 3)))
    odd = rng.random(n) < 0.1
    d[odd, :3] = rng.choice([np.nan, np.inf, -np.inf, 0.0, 1.0], size=(int(odd.sum()), 3))
    o[odd & (rng.random(n) < 0.3), 0] = np.nan
    print("rays with NaN, infinite and zero components among others", flush=True)
    tri, t, _, _ = orc.trace(T, *v, o, d, 1e-4)
    gtri, gt, _, _ = [x.cpu().numpy() if x is not None else None for x in api.trace_closest(DT, o, d, 1e-4)]
    assert np.array_equal(gtri[~odd], tri[~odd])
    assert np.array_equal(gt[~odd].view(np.uint32), t[~odd].view(np.uint32))


def test_captured_launch_has_a_wave_per_window(cuda, trees):
    # more rays than a counter's launch starts at: a captured call records no allocation
    torch = cuda
    DT, n = trees[2], 700001
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    rays = [(torch.rand((n, 4), device="cuda", generator=g) * 2 - 1, torch.randn((n, 4), device="cuda", generator=g))
            for _ in range(3)]
    o, d = rays[0][0].clone(), rays[0][1].clone()
    api.trace_closest(DT, o, d, 1e-4)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        tri, t, uv, _ = api.trace_closest(DT, o, d, 1e-4)
    for a, b in rays:
        print("replay", flush=True)
        o.copy_(a)
        d.copy_(b)
        graph.replay()
        torch.cuda.synchronize()
        etri, et, euv, _ = api.trace_closest(DT, a, b, 1e-4)
        assert torch.equal(tri, etri) and torch.equal(t, et) and torch.equal(uv, euv)
