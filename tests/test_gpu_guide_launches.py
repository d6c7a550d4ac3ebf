"""guide_launches counts the inference launches of a guided run: bounces 0 .. depth - 2 of every chunk sample
a continuation, of which the guide takes the first guided_bounces (0: all)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth,bounces,chunk,want", [(5, 0, 0, 4), (5, 2, 0, 2), (1, 0, 0, 0), (5, 0, 1 << 14, 16),
                                                      (3, 9, 1 << 14, 8)])
def test_launches_are_counted(ctx, cornell, depth, bounces, chunk, want):
    from banshee_amd import hip
    s = hip.Scene(ctx, cornell)
    old = ctx.tuning()
    try:
        ctx.set_tuning(paths_per_chunk=chunk)
        g = hip.Guide(ctx, 3, guided_bounces=bounces)
        s.render_guided(128, 128, 2, depth, 7, guide=g)
        st = ctx.stats()
        assert st["guide_launches"] == want
        assert (st["guide_ms"] > 0) == (want > 0) and (st["guide_rows"] > 0) == (want > 0)
        s.bake_sh_guided(np.float32([[1.0, 1.0, 1.0]] * 256), 256, 2, depth, 7, guide=g)
        assert ctx.stats()["guide_launches"] == want
        s.render(128, 128, 2, depth, 7)
        assert ctx.stats()["guide_launches"] == 0
    finally:
        ctx.set_tuning(**old)
