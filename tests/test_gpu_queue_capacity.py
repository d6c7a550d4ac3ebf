"""Bounces that queue nearly every ray their paths may: normal-mapped surfaces under an environment light.

The reference's estimator traces two MIS rays per light from a normal-mapped vertex, and an
environment light's pdf passes for almost all of them, so with the extension ray a bounce queues 2.9
closest-hit rays per path. A flat normal map leaves the shading normal as it is, so every camera
sample is that of the same floor without the map, whose vertices trace one MIS ray."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _floors(kind, bump):
    """(normal-mapped, plain) floor under a sky; one light."""
    from banshee_amd.scenes import Scene, env_map, floor_under
    plain = floor_under([kind, 0, 0, 0, 0, 0, 0, 0.8, 1.0], env=env_map(32, 16))
    plain.uvs = np.float32([[0, 0], [2, 0], [2, 2], [0, 2]])
    plain.tri_uv = plain.tri_v.copy()
    mapped = Scene(**{k: getattr(plain, k) for k in plain.__dataclass_fields__})
    texel = np.float32([0.5, 0.5, 1.0]) if not bump else np.float32([0.6, 0.45, 0.9])
    mapped.textures = [np.tile(texel, (4, 4, 1))]
    mapped.normal_maps = np.zeros(plain.materials.shape[0], np.int32)
    return mapped, plain


def _render(ctx, sc, chunk=0, refill=0):
    from banshee_amd import hip
    old = ctx.tuning()
    try:
        ctx.set_tuning(paths_per_chunk=chunk, refill_lanes=refill, lanes=1)
        s = hip.Scene(ctx, sc)
        ps = s.render(64, 64, 4, 3, 5, per_sample=True)[3]
        return ps, ctx.launch_stats()
    finally:
        ctx.set_tuning(**old)


@pytest.mark.parametrize("refill", [0, -1])
@pytest.mark.parametrize("kind", ["env", "envis"])
def test_flat_map_under_a_sky_is_no_map(ctx, kind, refill):
    from banshee_amd.scenes import ENV_LIGHT, ENV_LIGHT_IS
    mapped, plain = _floors(ENV_LIGHT if kind == "env" else ENV_LIGHT_IS, False)
    a, la = _render(ctx, mapped, refill=refill)
    b, lb = _render(ctx, plain, refill=refill)
    n = 64 * 64 * 16
    print(f"closest-hit rays per path of the second launch: {la[1]['rays_closest'] / n:.3f}, {lb[1]['rays_closest'] / n:.3f}")
    if kind == "env":   # the importance-sampled light's pdf is small away from the sun
        assert la[1]["rays_closest"] > 2.5 * n
    # the map's normalisations round, so a sample at a threshold may fall to its other side
    close = np.all(np.abs(a - b) <= 1e-5 + 1e-4 * np.abs(b), axis=-1)
    assert close.mean() >= 0.99, close.mean()


def test_full_queues_do_not_depend_on_the_chunk(ctx):
    from banshee_amd.scenes import ENV_LIGHT
    mapped, _ = _floors(ENV_LIGHT, True)
    a, la = _render(ctx, mapped)
    b, lb = _render(ctx, mapped, chunk=4096)
    assert la[1]["rays_closest"] == lb[1]["rays_closest"] > 2.5 * 64 * 64 * 16
    np.testing.assert_array_equal(a, b)
