// Sizes of the wavefront's per-path NEE slots and ray queues. Plain C++, so that the host tests compile it too.
#pragma once

#include <cstddef>

namespace bsh {

// log2 of a path's NEE slots when a vertex samples `lights` lights: light j's shadow ray is slot 2 j and
// its MIS ray slot 2 j + 1, and with normal maps (the reference's estimator, which may trace a second
// MIS ray per light) that second ray is slot 2 lights + 2 j + 1. A power of two, since a ray's owner
// is path << shift | slot; even slots are shadow rays, odd ones MIS rays.
constexpr int nee_slot_shift(int lights, bool normal_maps)
{
    int shift = 1;
    while ((1 << shift) < (normal_maps ? 4 : 2) * lights) ++shift;
    return shift;
}

// Most rays of one path in a bounce's queues: the extension ray and every odd slot are closest-hit rays,
// every even slot an any-hit ray. The queues hold that many per path of a chunk (a bounce may
// emit them all: one environment light over normal-mapped surfaces makes nearly three closest-hit
// rays per path).
constexpr size_t closest_rays_per_path(int shift) { return 1 + ((size_t)1 << shift) / 2; }
constexpr size_t any_rays_per_path(int shift) { return ((size_t)1 << shift) / 2; }

}  // namespace bsh
