"""Boxes of a tree over triangles whose corners are not numbers: a node's box passes
over them, and is not a number itself where it holds nothing else.  Against the
union of the leaves in numpy."""
import numpy as np
import pytest

from eos_amd import scenes

pytestmark = pytest.mark.gpu


def _soup(n, seed, bad):
    rng = np.random.default_rng(seed)
    v = rng.random((n, 3, 3)).astype(np.float32)
    v[bad] = np.nan
    return scenes.SceneData(v, np.tile(np.float32([0, 0, 1]), (n, 3, 1)), np.zeros(n, np.int32),
                            scenes.make_material((0.5, 0.5, 0.5), (0.5, 0.5, 0.5), 8)[None],
                            scenes.make_lights([(2.0, 3.0, 3.0)]),
                            scenes.make_camera((0.5, 0.5, 3.0), (0.5, 0.5, 0.5), 60.0, 16, 16), 0)


# runs of bad triangles below and across the leaf kernel's quads, waves and
# workgroups (1,024 leaves), and nothing but bad triangles
@pytest.mark.parametrize("n,first,count", [(2, 0, 2), (64, 10, 10), (700, 3, 600), (5000, 100, 2500)])
def test_boxes_of_triangles_that_are_not_numbers(n, first, count):
    from eos_amd import _lib as E
    s = _soup(n, n, slice(first, first + count))
    g = E.Scene(s, leaf_max=1)
    ibox, perm, kchild = g.debug_read("ibox"), g.debug_read("perm"), g.debug_read("kchild")
    v = s.verts[perm]
    lo, hi = np.fmin.reduce(v, axis=1), np.fmax.reduce(v, axis=1)
    want = np.full((n - 1, 6), np.nan, np.float32)
    done = np.zeros(n - 1, bool)
    stack = [0]
    while stack:
        i = stack[-1]
        todo = [c for c in kchild[i] if c >= 0 and not done[c]]
        if todo:
            stack += todo
            continue
        for c in kchild[i]:
            a, b = (want[c, :3], want[c, 3:]) if c >= 0 else (lo[~c], hi[~c])
            want[i, :3], want[i, 3:] = np.fmin(want[i, :3], a), np.fmax(want[i, 3:], b)
        done[i] = True
        stack.pop()
    assert np.isnan(want).any()
    assert np.array_equal(ibox, want, equal_nan=True)
    # the same tree from a batched build
    other, again = E.Scene(_soup(333, 1, slice(0, 5)), build=False), E.Scene(s, build=False)
    E.build_batch([other, again], leaf_max=1)
    assert np.array_equal(again.debug_read("nodes"), g.debug_read("nodes"), equal_nan=True)
