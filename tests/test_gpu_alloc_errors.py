"""A device allocation that fails is reported once, by the call that needed it, and leaves no error in
the runtime for a later call to report."""

from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from mnrt_amd import api, native as N
from helpers import f4

pytestmark = pytest.mark.gpu


def test_build_after_one_that_found_no_memory(cuda):
    torch = cuda
    rng = np.random.default_rng(0)
    c = rng.uniform(-1, 1, (1000000, 3))
    v = [api.dev(f4(c + rng.normal(scale=0.001, size=c.shape))) for _ in range(3)]
    small = [a[:500].contiguous() for a in v]
    want = api.build_tri(*small).nodes_host()
    p = api.default_params(0)
    p.small_node_max = 1  # a workspace of 6 GB, before it grows
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    rest = torch.empty(torch.cuda.mem_get_info()[0] - (3 << 30), dtype=torch.uint8, device="cuda")
    print("a build without room", flush=True)
    with ThreadPoolExecutor(1) as other:  # a thread of its own: it keeps no workspace of earlier builds
        with pytest.raises(N.MnrtError, match=r"\(-3\)"):
            other.submit(api.build_tri, *v, p).result()
        del rest
        torch.cuda.empty_cache()
        print("and one with room", flush=True)
        assert np.array_equal(other.submit(api.build_tri, *small).result().nodes_host(), want)
