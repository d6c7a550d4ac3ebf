"""The autotuner's own sweep times the automatic trace grid too, and keeps it where no other is faster.

The chunks of this run hold fewer rays than the smallest candidate's grid has lanes (2 workgroups per CU
on 256 CUs: 131,072), so every candidate launches the same kernels and the automatic grid is kept, up to
differences of more than 1 % between single runs (hence three tries)."""
import pytest

pytestmark = pytest.mark.gpu


def test_the_automatic_grid_is_a_candidate(ctx, terrain100k):
    from banshee_amd import hip
    s = hip.Scene(ctx, terrain100k)
    old = ctx.tuning()
    try:
        ctx.set_tuning(lanes=1)
        job = hip.BatchJob(s, "render", width=512, height=512, img_grid=2, max_depth=4, seed=3)
        got = []
        while len(got) < 3 and 0 not in got:
            best, ms = ctx.autotune([job], paths=[1 << 15])
            assert best["paths_per_chunk"] == 1 << 15 and best["lanes"] == 1 and ms > 0
            got.append(best["trace_blocks_per_cu"])
        assert got[-1] == 0, got
        assert ctx.tuning()["trace_blocks_per_cu"] == 0
        with pytest.raises(hip.BshError, match="candidate"):
            ctx.autotune([job], paths=[1 << 15], blocks=[0])
    finally:
        ctx.set_tuning(**old)
