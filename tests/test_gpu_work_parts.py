"""Queue sizes at the edges of the trace kernel's work split.

The refill kernel deals a launch's ray queue to 16 work counters in runs of 2048 entries, and its
grid shrinks with the chunk; refill_lanes = -1 traces the same queue in 64-ray batches from one
counter. Every camera sample has to come out the same, bit for bit, whatever the split."""
import numpy as np
import pytest

from banshee_amd import hip

pytestmark = pytest.mark.gpu


# pixels x samples: 1 path, a wave +- 1, a run +- 1, all 16 parts' first runs +- 1 and the second
# round's remainder in a middle part
@pytest.mark.parametrize("w,h", [(1, 1), (63, 1), (65, 1), (89, 23), (64, 32), (683, 3), (151, 217), (128, 256),
                                 (993, 33), (257, 271)])
@pytest.mark.parametrize("claim", [0, 96])
def test_samples_do_not_depend_on_the_queue_split(ctx, cornell, terrain100k, w, h, claim):
    old = ctx.tuning()
    try:
        for sc in (cornell, terrain100k):
            s = hip.Scene(ctx, sc)
            ctx.set_tuning(refill_lanes=-1)
            ref = s.render(w, h, 1, 4, 11, per_sample=True)
            rays = s.stats()["rays_closest"], s.stats()["rays_any"]
            ctx.set_tuning(claim_rays=claim)
            got = s.render(w, h, 1, 4, 11, per_sample=True)
            assert (s.stats()["rays_closest"], s.stats()["rays_any"]) == rays
            np.testing.assert_array_equal(got[3], ref[3])
    finally:
        ctx.set_tuning(**{k: old[k] for k in ("paths_per_chunk", "trace_blocks_per_cu", "use_graph", "refill_lanes",
                                               "claim_rays", "lanes")})
