"""Ray queries whose box entry distances are enormous or infinite and negative.

bsh_ray takes any tmin, so an entry distance max(slabs, tmin) may be any float or -inf: rays that start
past the scene and run away from it on all axes, with an interval that reaches behind them. Such a
node's leaf and empty children must not be taken for internal ones. The plain loop
(bsh_intersect_count) selects children by their counts alone, and every hit has to agree with
it bit for bit."""
import numpy as np
import pytest

from banshee_amd import hip
from banshee_amd.scenes import cornell_box, terrain_for_tris
from test_gpu_query_refill import check

pytestmark = pytest.mark.gpu


def rays_for(sc, n, far, small, seed):
    """Origins `far` away on every axis or in the scene, directions of length about `small` or 1."""
    r = np.random.default_rng(seed)
    lo, hi = sc.verts.min(0), sc.verts.max(0)
    o = r.uniform(lo, hi, (n, 3))
    d = np.where(r.random((n, 3)) < 0.5, -1.0, 1.0) * r.uniform(0.3, 1.0, (n, 3))
    k = np.arange(n)
    out = k % 3 == 1                               # outside, the scene behind (or ahead for k % 2)
    o[out] += far * np.where(k[out] % 2 == 1, 1.0, -1.0)[:, None] * np.sign(d[out])
    d[out] *= small
    tmin = np.array([-np.inf, -3.4e38, -1e38, -1e37, -1.0, 0.0])[k // 3 % 6]
    tmax = np.array([np.inf, 3e38, 1e6, 0.0, -1e-3])[k // 18 % 5]
    return np.concatenate([o, tmin[:, None], d, tmax[:, None]], 1).astype(np.float32)


# far / small: entry distances of -1e38, of -inf (overflowed 1 / d products), and of the ordinary range
@pytest.mark.parametrize("far,small", [(1e18, 1e-20), (1e19, 1e-20), (1e19, 1e-19), (1e20, 1.0), (3e38, 1.0), (100.0, 1.0)])
@pytest.mark.parametrize("quantized", [True, False])
@pytest.mark.parametrize("max_leaf", [1, 8])
def test_far_negative_intervals(ctx, far, small, quantized, max_leaf):
    for sc in (cornell_box(), terrain_for_tris(3000, seed=5)):
        s = hip.Scene(ctx, sc, width=4, quantized=quantized, max_leaf=max_leaf)
        assert s.info()["width"] == 4 and s.info()["quantized"] == quantized
        prim = check(s, rays_for(sc, 6000, far, small, 9))
        inside = np.arange(6000) % 3 != 1
        assert (prim[inside] >= 0).mean() > 0.1


def test_probe_rays_that_reach_behind_their_probes(ctx):
    """A probe job's tmin may be negative or -inf too: the bake equals the one traced in whole batches,
    and a captured batch is not replayed for a job whose tmin takes it to the other trace kernel."""
    s = hip.Scene(ctx, terrain_for_tris(3000, seed=5))
    p = np.float32([[0.0, 8.0, 0.0], [3.0, 6.0, -2.0], [100.0, 90.0, 80.0]])
    old = ctx.tuning()
    try:
        for tmin in (-np.inf, -3e38, -1e36, -1.0):
            ctx.set_tuning(refill_lanes=-1)
            ref = s.bake_sh(p, 64, 2, 3, 5, tmin=tmin)
            ctx.set_tuning()
            np.testing.assert_array_equal(s.bake_sh(p, 64, 2, 3, 5, tmin=tmin)[0], ref[0])
        replayed = []
        for tmin in (0.0, 0.0, -np.inf, 0.0):
            j = hip.BatchJob(s, "bake", probes=p, rays_per_probe=64, lmax=2, max_depth=3, seed=5, tmin=tmin)
            ctx.batch_run([j], tuning={"use_graph": 1})
            replayed.append(ctx.stats()["graph_replayed"])
        assert replayed == [0, 1, 0, 0]
    finally:
        ctx.set_tuning(**old)
