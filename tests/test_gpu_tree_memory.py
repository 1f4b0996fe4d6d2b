"""Device memory of ray-tree frames: per level of the tree what its rays need, with two
levels' surfaces in a single frame (one is shaded while the next is set up) and one
in each of the frames in flight."""
import pytest

from eos_amd import scenes

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _slot_bytes(w, h, depth, lights, two):
    """The buffers of one frame, without the fixed ones (counters, overflow stacks)."""
    npix, n_ids = w * h, ((w + 7) // 8) * ((h + 7) // 8) * 64
    cap = [npix << lev for lev in range(depth + 1)]
    surfaces = max(cap[::2]) + max(cap[1::2], default=0) if two else max(cap)
    return (16 * n_ids + (2 * 32 + 16) * max(cap) + (32 + lights) * surfaces + (16 * (depth + 1) + 1) * npix
            + 36 * sum(cap) + n_ids // 8)


@pytest.mark.parametrize("depth", [0, 1, 2, 3])
def test_tree_frames(depth):
    import numpy as np
    import torch
    from eos_amd import _lib as E
    w, h, aa = 1365, 767, 2
    print(f"tree memory depth={depth}", flush=True)
    s = scenes.glass(w, h, level=2, depth=depth)
    lights = len(s.lights)
    img = torch.zeros((h, w, 4), dtype=torch.uint8, device="cuda")
    E.Scene(scenes.glass(32, 32, level=2, depth=1)).render(aa_samples=aa)    # the library's own start
    g = E.Scene(s)
    g.render(camera=scenes.glass(32, 32, level=2, depth=depth).camera)      # fixed buffers of slot 0
    slack = 24 * 2 * MIB                             # each buffer rounded up by the allocator
    stacks = 2 * 256 * 16 * 64 * 80 * 4              # overflow stacks of slot 1: 16 waves per CU, twice

    def taken(aa_samples):
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        g.render_device(s.camera, depth, img.data_ptr(), aa_samples=aa_samples)
        return before - torch.cuda.mem_get_info()[0]

    single = taken(0)
    assert single <= _slot_bytes(w, h, depth, lights, True) + slack, single
    first = img.cpu().numpy().copy()
    flight = taken(aa)                          # a second slot, of frames on one stream
    assert flight <= _slot_bytes(w, h, depth, lights, False) + 16 * w * h + stacks + slack, flight
    g.render_device(s.camera, depth, img.data_ptr())
    assert np.array_equal(first, img.cpu().numpy())
