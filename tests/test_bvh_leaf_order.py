"""The 4-wide tree's leaf order (CPU only): what the traversal's triangle bit masks assume.

In every node the leaf children come before the internal ones and the empty slots come last, the
leaf children's triangles are consecutive from the first slot's ref on, and the quantised node's
leaf bits (word 11) hold one low bit per triangle in the child's byte.
"""
import numpy as np
import pytest

from banshee_amd import hip
from banshee_amd.scenes import cornell_box, terrain_for_tris

pytestmark = pytest.mark.skipif(not __import__("os").path.exists(hip.LIB_PATH), reason="library not built")


@pytest.mark.parametrize("max_leaf", [1, 2, 4, 7, 8, 20])
@pytest.mark.parametrize("make", [cornell_box, lambda: terrain_for_tris(3000, seed=3)])
def test_leaf_children_first_and_consecutive(make, max_leaf):
    sc = make()
    tv = sc.verts[sc.tri_v].reshape(-1, 9).astype(np.float32)
    nq, order, w, _ = hip.bvh_build_host(tv, width=4, quantized=True, max_leaf=max_leaf)
    assert w == 4 and nq.shape[1] == 16 and sorted(order.tolist()) == list(range(len(tv)))
    u = nq.view(np.uint32)
    cnt = np.stack([((u[:, 10] >> (8 * c)) & 255).astype(np.uint8).view(np.int8) for c in range(4)], -1).astype(int)
    ref, bits = nq.view(np.int32)[:, 12:16], u[:, 11]
    kind = np.where(cnt > 0, 0, np.where(cnt == 0, 1, 2))
    assert np.all(np.diff(kind, axis=1) >= 0)
    assert cnt.max() <= min(max_leaf, 8)
    for k in range(len(nq)):
        nleaf = int((kind[k] == 0).sum())
        assert np.array_equal(ref[k, :nleaf], ref[k, 0] + np.cumsum(cnt[k, :nleaf]) - cnt[k, :nleaf])
        want = sum(((1 << cnt[k, c]) - 1) << (8 * c) for c in range(nleaf))
        assert int(bits[k]) == want
        inner = ref[k][kind[k] == 1]
        assert np.all(np.diff(inner) > 0) and np.all(inner > k)
