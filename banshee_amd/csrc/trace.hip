// Ray-query kernels: the Intersectable slot (closest / any hit) over caller ray buffers.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "internal.h"
#include "trace_core.h"

namespace bsh {

constexpr int kTraceBlock = 256;

// Ray queries on a 4-wide BVH: the refill loop of trace_core.h, one wave per workgroup over its own
// `span` consecutive rays, so a wave replaces finished rays without any shared counter and the
// hardware's workgroup dispatch balances the waves. Bound by VALU issue and node latency as the
// wavefront's trace kernel; 4 KB of LDS and 64 VGPRs allow 32 waves per CU, where one thread per
// ray with its whole stack in LDS (48 KB per 256 rays) held 12 and ended each wave with its
// slowest ray. 2M random rays, 3.08M triangles: 2017 -> 415 us; 700,001 shadow rays, 500k
// triangles: 388 -> 136 us; 1000 camera rays, 34 triangles: 14.2 -> 10.1 us.
constexpr int kQueryLds = 16;       // LDS stack entries per lane (4 KB per wave), deeper ones in scratch
// Idle lanes that trigger a refill. Measured (us, 2M random rays on 3.08M triangles at span 192):
// 8 396, 16 395, 24 397, 32 406, 48 447, 56 482; without a claim a refill costs little.
constexpr int kQueryRefill = 16;
// Rays per wave: one per lane until the waves of 64 rays outnumber what the GPU holds at once
// (24 waves on each of 256 CUs), then 128 or 192, so that fewer lanes wait for a wave's last rays.
// Measured with 64 / 128 / 192 / 256 / 384 (us): 100,003 rays 60 / 68 / 79 / 87 / 105; 500,003
// 104 / 91 / 98 / 115 / 135; 700,001 168 / 143 / 146 / 156 / 200; 2M random 499 / 401 / 395 / 388 /
// 378; 2M camera rays 359 / 359 / 351 / 369 / 436.
static uint32_t query_span(uint32_t n)
{
    const uint32_t resident = 64u * 24u * 256u;
    return 64u * std::min(3u, std::max(1u, n / resident + (n % resident != 0u)));
}

// Stack entries past kQueryLds, in the lane's private memory.
struct ScratchOvf
{
    uint32_t* p;
    __device__ __forceinline__ uint32_t& at(int i) const { return p[i]; }
};

template <bool kAny, bool kQ>
__global__ __launch_bounds__(64, 8) void k_query4(const float4* __restrict__ nodes, const float4* __restrict__ tris,
                                                  const bsh_ray* __restrict__ rays, uint32_t n, uint32_t span,
                                                  bsh_hit* __restrict__ hits, int32_t* __restrict__ occ)
{
    __shared__ __align__(16) uint32_t stk[kQueryLds * 64];
    uint32_t deep[kMaxStack4 - kQueryLds];
    const ScratchOvf ovf{deep};
    const int lane = threadIdx.x;
    uint32_t rb = blockIdx.x * span;
    const uint32_t re = min(n, rb + span);
    uint32_t idx = 0, nv = 0, tv = 0;
    bool active = false;
    LaneRay r{};
    for (;;)
    {
        const unsigned long long idle = __ballot(!active);
        const uint32_t nidle = (uint32_t)__popcll(idle);
        if (rb < re && (nidle >= (uint32_t)kQueryRefill || nidle == 64u))
        {
            if (!active)
            {
                const uint32_t q = rb + (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
                if (q < re)
                {
                    idx = q;
                    const float4* r4 = reinterpret_cast<const float4*>(rays);
                    start_ray<64>(r, stk, gload(r4, 2 * (size_t)q), gload(r4, 2 * (size_t)q + 1));
                    active = true;
                }
            }
            rb += min(re - rb, nidle);
        }
        if (__ballot(active) == 0ull) break;
        if (!active) continue;
        if (!step4<false, kQ, false, true, kQueryLds, 64>(r, kAny, nodes, tris, stk, ovf, nv, tv)) continue;
        const bool h = r.prim >= 0;
        if (kAny && occ) occ[idx] = h ? 1 : 0;
        if (hits)
        {
            bsh_hit o;
            o.prim = r.prim;
            o.t = h ? r.tcur : 0.f;
            o.b1 = r.b1;
            o.b2 = r.b2;
            hits[idx] = o;
        }
        active = false;
    }
}

// One thread per ray: binary BVHs, and every layout in counting mode.
template <bool kAny, bool kCount>
__global__ __launch_bounds__(kTraceBlock) void k_intersect(SceneDev s, const bsh_ray* __restrict__ rays, uint32_t n,
                                                           bsh_hit* __restrict__ hits, int32_t* __restrict__ occ,
                                                           uint32_t* __restrict__ visits)
{
    // whole stack in LDS: 32 entries x 4 B x 256 threads = 32 KB, 48 KB where a 4-wide BVH is traced
    __shared__ uint32_t stk[(kCount ? kMaxStack4 : kMaxStack) * kTraceBlock];
    uint32_t i = blockIdx.x * kTraceBlock + threadIdx.x;
    if (i >= n) return;
    const float4* r4 = reinterpret_cast<const float4*>(rays);
    float4 a = r4[2 * i], b = r4[2 * i + 1];
    TraceResult res;
    TraceCounts cnt{0u, 0u};
    bool h = kCount && s.width == 4
                 ? traverse4<kAny, kCount, kMaxStack4>(s, mk(a.x, a.y, a.z), mk(b.x, b.y, b.z), a.w, b.w,
                                                       stk + threadIdx.x, kTraceBlock, res, cnt, nullptr, 0)
                 : traverse<kAny, kCount>(s, mk(a.x, a.y, a.z), mk(b.x, b.y, b.z), a.w, b.w, stk + threadIdx.x,
                                          kTraceBlock, res, cnt);
    if (kAny && occ) occ[i] = h ? 1 : 0;
    if (hits)
    {
        bsh_hit o;
        o.prim = h ? res.prim : -1;
        o.t = h ? res.t : 0.f;
        o.b1 = h ? res.b1 : 0.f;
        o.b2 = h ? res.b2 : 0.f;
        hits[i] = o;
    }
    if (kCount && visits)
    {
        visits[2 * i] = cnt.nodes;
        visits[2 * i + 1] = cnt.tris;
    }
}

bsh_status launch_intersect(bsh_scene* s, const bsh_ray* rays, size_t n, int any, bsh_hit* hits, int32_t* occ,
                            uint32_t* visits, hipStream_t st)
{
    if (!s) return fail(BSH_ERR_INVALID, "intersect: NULL scene");
    if (!s->committed) return fail(BSH_ERR_STATE, "intersect: scene not committed");
    if (n == 0) return BSH_OK;
    if (!rays || (!hits && !occ)) return fail(BSH_ERR_INVALID, "intersect: NULL buffer");
    if (n > 0xffffffffull - kTraceBlock) return fail(BSH_ERR_INVALID, "intersect: too many rays");
    BSH_HIP(hipSetDevice(s->ctx->device));
    dim3 grid((uint32_t)((n + kTraceBlock - 1) / kTraceBlock));
    SceneDev d = s->dev();
    if (!visits && d.width == 4)
    {
        const uint32_t span = query_span((uint32_t)n);
        const dim3 g((uint32_t)((n + span - 1) / span)), b(64);
        if (any && d.qnodes) hipLaunchKernelGGL((k_query4<true, true>), g, b, 0, st, d.nodes, d.tris, rays, (uint32_t)n, span, hits, occ);
        else if (any) hipLaunchKernelGGL((k_query4<true, false>), g, b, 0, st, d.nodes, d.tris, rays, (uint32_t)n, span, hits, occ);
        else if (d.qnodes) hipLaunchKernelGGL((k_query4<false, true>), g, b, 0, st, d.nodes, d.tris, rays, (uint32_t)n, span, hits, occ);
        else hipLaunchKernelGGL((k_query4<false, false>), g, b, 0, st, d.nodes, d.tris, rays, (uint32_t)n, span, hits, occ);
    }
    else if (visits)
    {
        if (any) hipLaunchKernelGGL((k_intersect<true, true>), grid, dim3(kTraceBlock), 0, st, d, rays, (uint32_t)n, hits, occ, visits);
        else hipLaunchKernelGGL((k_intersect<false, true>), grid, dim3(kTraceBlock), 0, st, d, rays, (uint32_t)n, hits, occ, visits);
    }
    else
    {
        if (any) hipLaunchKernelGGL((k_intersect<true, false>), grid, dim3(kTraceBlock), 0, st, d, rays, (uint32_t)n, hits, occ, visits);
        else hipLaunchKernelGGL((k_intersect<false, false>), grid, dim3(kTraceBlock), 0, st, d, rays, (uint32_t)n, hits, occ, visits);
    }
    BSH_HIP(hipGetLastError());
    return BSH_OK;
}

}  // namespace bsh
