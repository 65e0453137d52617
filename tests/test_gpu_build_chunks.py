"""Builds whose root has as many elements as a node's wave sums its chunks' counts in one pass (64 chunks
of 64 waves of 64 slots), and one more.  Node words and references equal the oracle's."""

import numpy as np
import pytest

from mnrt_amd import api
from helpers import f4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64 ** 3, 64 ** 3 + 1])
@pytest.mark.parametrize("kind", [0, 1])
def test_chunk_passes(orc, cuda, kind, n):
    rng = np.random.default_rng(n + kind)
    c = rng.uniform(-1.0, 1.0, (n, 3))
    v = [f4(c + rng.normal(scale=0.003, size=c.shape)) for _ in range(3)] if kind == 0 else [f4(c)]
    print(f"kind {kind} n {n}", flush=True)
    dt = api.build_tri(*v) if kind == 0 else api.build_points(v[0])
    cuda.cuda.synchronize()
    ot = orc.build(kind, *v, small_max=64 if kind == 0 else 32)
    assert np.array_equal(dt.nodes_host(), ot.nodes)
    assert np.array_equal(dt.refs_host(), ot.refs)
