"""Photon trees much deeper than a balanced one: queries walk their node words although a hierarchy is
there, and give what the hierarchy gives, bit for bit, on both sides of the line."""

import pytest
import torch

from mnrt_amd import api, native as N

pytestmark = pytest.mark.gpu


def _f4(x):
    return torch.cat([x, torch.zeros((x.shape[0], 1))], dim=1).float().contiguous().cuda()


def _bits(t):
    return t.contiguous().view(torch.int32)


def _with_level(tree, level):
    w = api.DeviceTree(N.KIND_POINT, N.Tree.from_buffer_copy(tree.t), batch=tree)  # a view: releases nothing
    w.t.max_level = level
    return w


def _unit(g, n):
    return torch.nn.functional.normalize(torch.randn((n, 3), generator=g), dim=1)


@pytest.mark.parametrize("n,q", [(1, 70), (255, 600), (30000, 9000)])
def test_both_sides_of_the_line(cuda, n, q):
    g = torch.Generator(device="cpu").manual_seed(n)
    z = torch.randn((n, 3), generator=g)
    at = (z * z * z * 0.05).clamp(-1, 1)
    pos = _f4(at)
    tree = api.build_points(pos, api.default_params(N.KIND_POINT, [-1, -1, -1, 1, 1, 1], 0.2))
    api.attach_photon_records(tree, pos, _f4(z.abs()), _f4(_unit(g, n)))
    assert tree.t.owns_qnodes & N.QNODES_BOXES
    qp = _f4(at.repeat(q // n + 1, 1)[:q] + 0.002 * torch.randn((q, 3), generator=g))
    rest = [_f4(_unit(g, q)), _f4(_unit(g, q)), torch.ones((q, 4), device="cuda"), torch.rand((q, 4), generator=g).cuda()]
    grad = torch.rand((q, 4), generator=g).cuda()
    line = n.bit_length() + 17
    print(f"n {n}: {tree.t.max_level} levels, line {line}", flush=True)
    assert n < 30000 or tree.t.max_level > 30
    out = []
    for level in (line, line + 1):
        t = _with_level(tree, level)
        print(f"queries at level {level}", flush=True)
        r = api.knn_gather(t, 50, 0.2, qp, *rest, want_nbr=True, want_r2=True, want_irr=True, want_count=True)
        back = api.knn_gather_bwd(t, 50, 0.2, qp, *rest, grad, r["r2"], r["count"])
        out.append([r[c] for c in ("rad", "nbr", "r2", "irr", "count")] + [api.knn_radii(t, 50, 0.2, qp), *back])
    for x, y in zip(*out):
        assert torch.equal(_bits(x), _bits(y))
