"""Device memory that a scene's first small query takes: by its rays, not by its launch."""
import numpy as np
import pytest

from eos_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["nearest", "occluded"])
@pytest.mark.parametrize("n", [1, 1000, 3000])
def test_first_query(n, mode):
    import torch
    from eos_amd import _lib as E
    rng = np.random.default_rng(n)
    o, d = rng.normal(size=(n, 3)).astype(np.float32), rng.normal(size=(n, 3)).astype(np.float32)
    warm = E.Scene(scenes.config_a(16, 16))
    warm.trace_rays(o, d, mode)                     # the library's own start
    g = E.Scene(scenes.config_a(16, 16))
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    g.trace_rays(o, d, mode)
    taken = before - torch.cuda.mem_get_info()[0]
    # stacks of at most 80 entries per ray, rays, records and hits of 88 bytes, each of
    # the five buffers rounded up by the allocator (2 MiB)
    assert taken <= (320 + 88) * (n + 64) + 5 * (2 << 20), taken
