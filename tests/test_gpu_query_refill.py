"""Ray queries through the refill loop against the one-thread-per-ray traversal.

bsh_intersect_count traces with the plain loop (IEEE division in the triangle test, one conversion
and fma per box plane); bsh_intersect_closest / _any use the refill loop's forms of the same
arithmetic, so every hit has to agree bit for bit: ray counts at the edges of a wave and of the
rays-per-wave rule, closest and any hit, both 4-wide layouts, rays with zero direction components,
infinite and tiny intervals, and scenes whose determinants are subnormal, huge or zero."""
import numpy as np
import pytest

from banshee_amd import hip
from banshee_amd.scenes import terrain_for_tris

pytestmark = pytest.mark.gpu


def rays_for(sc, n, seed):
    r = np.random.default_rng(seed)
    lo, hi = sc.verts.min(0), sc.verts.max(0)
    o = r.uniform(lo, hi, (n, 3))
    d = r.normal(size=(n, 3))
    k = np.arange(n)
    d[k % 7 == 3, 0] = 0.0                        # slabs parallel to the ray
    d[k % 11 == 5, 1:] = 0.0
    d[k % 13 == 6] *= 1e-3                        # unnormalised directions
    d[k % 17 == 8] *= 1e4
    tmin = np.where(k % 5 == 1, 0.0, np.where(k % 5 == 2, -1.0, 0.01))
    tmax = np.where(k % 3 == 1, np.inf, np.where(k % 3 == 2, 1e6, np.linalg.norm(hi - lo) * r.uniform(0, 0.4, n)))
    return np.concatenate([o, tmin[:, None], d, tmax[:, None]], 1).astype(np.float32)


def check(s, rays):
    prim, hit = s.intersect(rays)
    p2, h2, _ = s.intersect_count(rays)
    np.testing.assert_array_equal(prim, p2)
    np.testing.assert_array_equal(hit.view(np.uint32), h2.view(np.uint32))
    occ, _ = s.intersect(rays, any_hit=True)
    p3, _, _ = s.intersect_count(rays, any_hit=True)
    np.testing.assert_array_equal(occ, (p3 >= 0).astype(np.int32))
    return prim


@pytest.mark.parametrize("quantized", [True, False])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 1000, 64 * 6144 - 1, 64 * 6144, 64 * 6144 + 1, 128 * 6144 + 65])
def test_matches_the_plain_loop(ctx, terrain100k, n, quantized):
    s = hip.Scene(ctx, terrain100k, width=4, quantized=quantized)
    prim = check(s, rays_for(terrain100k, n, n))
    assert n < 1000 or 0.05 < (prim >= 0).mean() < 1.0


# e1 x e2 scales with the square of the scene's size and det with the direction too: 1e-21 gives
# subnormal and zero determinants, 1e15 determinants near 2^126, past which 1 / det is subnormal
@pytest.mark.parametrize("scale", [1e-21, 1e-16, 1e-6, 1.0, 1e6, 1e15])
@pytest.mark.parametrize("max_leaf", [1, 8])
def test_scaled_scenes(ctx, scale, max_leaf):
    sc = terrain_for_tris(3000, seed=5)
    sc.verts = (sc.verts.astype(np.float64) * scale).astype(np.float32)
    s = hip.Scene(ctx, sc, max_leaf=max_leaf)
    rays = rays_for(sc, 20000, 3)
    rays[:, 3] *= np.float32(scale)
    check(s, rays)
