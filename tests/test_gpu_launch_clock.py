"""Launch durations from the kernels' clock stamps: on one lane the trace, inference and shade launches of a
run follow one another, so their sum is at most the run's time between events and most of it."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("guided,chunk", [(False, 0), (False, 1 << 16), (True, 0)])
def test_launch_durations_add_up(ctx, cornell, guided, chunk):
    from banshee_amd import hip
    s = hip.Scene(ctx, cornell)
    old = ctx.tuning()
    try:
        ctx.set_tuning(paths_per_chunk=chunk, lanes=1)
        g = hip.Guide(ctx, 3) if guided else None
        for _ in range(2):
            s.render_guided(256, 256, 4, 5, 7, guide=g) if guided else s.render(256, 256, 4, 5, 7)
        st, ls = ctx.stats(), ctx.launch_stats()
    finally:
        ctx.set_tuning(**old)
    parts = st["trace_ms"] + st["shade_ms"] + st["guide_ms"]
    assert len(ls) == 6 and all(l["trace_ms"] > 0 for l in ls)
    assert abs(sum(l["trace_ms"] for l in ls) - st["trace_ms"]) < 1e-6
    assert (st["guide_ms"] > 0) == guided and st["shade_ms"] > 0
    # 5 us: the two clocks' resolutions
    assert 0.5 * st["total_ms"] < parts < st["total_ms"] + 0.005
