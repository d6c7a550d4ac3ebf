// The 4-wide traversal loop with per-lane refill, shared by the wavefront's trace kernel
// (render.hip) and the ray queries (trace.hip).
//
// What bounds it is VALU issue: on the 3.08M-triangle terrain the vector pipes of a launch are
// busy 95 % of the time, about half of a wave's lanes active per instruction, because a wave
// runs a triangle test, a child sort and a node visit per iteration over whichever lanes need
// them. So the loop is written for few issue cycles, as measured on this part (cycles per wave
// instruction and SIMD): mul, add, sub, mov, and, or, integer add 2.5; fma, max, min, shifts,
// conversions, v_perm, compares and e64 selects 4.1-4.6, v_min_f64 the same; rcp 8.3; two e32
// selects on vcc back to back 45.
//  * Box planes: v_perm picks the entry (or exit) planes of two children by the direction's
//    sign and widens them to half floats in one instruction (a byte q as the subnormal half
//    q 2^-24), and v_fma_mix takes the halves as they are: 36 instructions for a node's 24
//    plane distances instead of 24 conversions, 24 fma, 3 compares and 6 selects.
//  * Which children are hit: the sign bits of (exit - entry), replicated to bytes by v_perm, are
//    and-ed with the node's leaf bits (the hit triangles) and turn the keys of children that are
//    missed, leaves or empty into sentinels with two instructions each.
//  * The sort: a key (entry distance) and its node index are the high and low word of a double,
//    so a compare-exchange is a v_min_f64 and a v_max_f64 instead of a compare and 4 selects.
//  * Leaf triangles: the node's leaves hold consecutive triangles, so the next one is found by
//    a popcount over the leaf bits instead of selects over four refs and counts.
//  * 1 / det: v_rcp and one Newton step (see rcp_exact).
// Per ray of that scene the loop issues 102 wave instructions instead of 153; with everything else
// as it was, the 1080p 64-sample frame took 249.0 ms against 283.9, a 4096-probe bake over 2M
// triangles 8.00 against 9.04, a batch of 16 scenes 13.1 against 14.4.
#pragma once

#include "scene_dev.h"

namespace bsh {

// 1.f / x with the same bits as the IEEE division, in 4 instructions instead of 10: one Newton
// step on the hardware reciprocal (error below 1 ulp) rounds correctly (P. Markstein,
// "Computation of elementary functions on the IBM RISC System/6000 processor", 1990; checked
// against the division for every mantissa at every exponent whose reciprocal is normal). A
// result that is not a normal number (x zero, subnormal, infinite, NaN or above 2^126) takes
// the division.
__device__ __forceinline__ float rcp_exact(float x)
{
    const float r = __builtin_amdgcn_rcpf(x);
    float q = __builtin_fmaf(__builtin_fmaf(-x, r, 1.f), r, r);
    if (!__builtin_amdgcn_classf(q, 0x108))   // +-normal
    {
        asm volatile("");   // keeps the division in the branch (it is otherwise executed by every lane)
        q = 1.f / x;
    }
    return q;
}

// Möller-Trumbore as intersect_face (bsh_math.h), the reciprocal by rcp_exact: the same bits.
__device__ __forceinline__ bool intersect_face_dev(f3 p1, f3 e1, f3 e2, f3 o, f3 d, float tmin, float tmax, float& t,
                                                   float& b1o, float& b2o)
{
    const f3 s1 = cross(d, e2);
    const float invd = rcp_exact(dot(s1, e1));
    const f3 dd = o - p1;
    const float b1 = dot(dd, s1) * invd;
    if (b1 < 0.f || b1 > 1.f) return false;
    const f3 s2 = cross(dd, e1);
    const float b2 = dot(d, s2) * invd;
    if (b2 < 0.f || b1 + b2 > 1.f) return false;
    const float tmp = dot(e2, s2) * invd;
    if (tmp > tmin && tmp <= tmax)
    {
        t = tmp;
        b1o = b1;
        b2o = b2;
        return true;
    }
    return false;
}

// A lane's ray and traversal state.
struct LaneRay
{
    f3 o, d;
    float ix, iy, iz, ox, oy, oz;   // 1 / d and o / d of the slab tests
    uint32_t selx, sely, selz;      // per axis: v_perm selector of the entry planes of children 0 and 1
    float tmin, tcur, b1, b2;
    int prim;
    uint32_t top;                   // the stack's top entry; the others in LDS, past kLds in `ovf`
    uint32_t spb;                   // byte offset of the lane's next free LDS slot
    uint32_t base, full, pend;      // the last visit's leaves: first triangle - 1, their bits, the hit ones left
    double k0, k1, k2, k3;          // its internal children: (entry distance, index)
};

constexpr uint32_t kSelLo = 0x0c010c00u, kSelHi = 0x0c050c04u;   // bytes 0, 1 of the second / first source
constexpr uint32_t kStackEnd = 0xffffffffu;                      // the stack's bottom entry
// Sentinel keys of the children that are not to be visited. With kAnyMin any tmin is allowed: the key
// of such a child is kKeyNone, above every float's bits (+inf among them) in the order of the doubles
// and as a float a NaN, which no comparison accepts. Without it tmin is at least kLeastMin, so
// every entry distance is, and the sentinel is formed by an fma: at least kKeyFar + kLeastMin, above
// kKeyMost, beyond which entry distances are culled. (With an entry distance of -1e38 or -inf the
// fma would give a leaf's key a value to be visited, as a node, at its first triangle's index.) The
// selecting form takes one instruction more per visit: 1080p frame 191.1 ms with the fma, 192.6
// with the selection, 700,001 shadow rays 156.7 / 157.6 us. The wavefront, whose tmin the host
// knows, takes the fma, the ray queries the selection.
constexpr uint32_t kKeyNone = 0x7f900000u;
constexpr float kKeyFar = 1.7014118e38f, kKeyMost = 1.5e38f, kLeastMin = -1e37f;

typedef _Float16 th2 __attribute__((ext_vector_type(2)));

// Visits `node`: the hit leaf triangles (pend) and the internal children's keys. kQ: GpuNodeQ
// nodes, else GpuNode4. kOne: `nodes` is the same for every lane and smaller than 4 GiB. kAnyMin: see
// kKeyNone.
template <bool kQ, bool kOne, bool kAnyMin>
__device__ __forceinline__ void visit4(LaneRay& r, const float4* nodes, uint32_t node)
{
    float tn[4], df[4];
    int ref[4];
    uint32_t cnts, leaf;
    if (kQ)
    {
        const float4* p = kOne ? reinterpret_cast<const float4*>(reinterpret_cast<const char*>(nodes) + (node << 6))
                               : nodes + 4 * (size_t)node;
        const float4 W0 = gload(p, 0);
        const int4 I1 = gload_i(p, 1), I2 = gload_i(p, 2);
        const int4 REF = gload_i(p, 3);
        ref[0] = REF.x; ref[1] = REF.y; ref[2] = REF.z; ref[3] = REF.w;
        cnts = (uint32_t)I2.z;
        leaf = (uint32_t)I2.w;
        // plane q of an axis is met at q (2^e / d) + (origin / d - o / d); the half-float
        // planes are q 2^-24, exactly, so the scale is 2^(e + 24) / d (exact: e is at most 36)
        const uint32_t ex = __float_as_uint(W0.w);
        const float sx = __builtin_amdgcn_ldexpf(r.ix, (int)(int8_t)(ex & 0xffu) + 24);
        const float sy = __builtin_amdgcn_ldexpf(r.iy, (int)(int8_t)((ex >> 8) & 0xffu) + 24);
        const float sz = __builtin_amdgcn_ldexpf(r.iz, (int)(int8_t)((ex >> 16) & 0xffu) + 24);
        const float bx = __builtin_fmaf(W0.x, r.ix, -r.ox), by = __builtin_fmaf(W0.y, r.iy, -r.oy),
                    bz = __builtin_fmaf(W0.z, r.iz, -r.oz);
        th2 nx[2], fx[2], ny[2], fy[2], nz[2], fz[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
        {
            const uint32_t qx = r.selx + 0x00020002u * h, qy = r.sely + 0x00020002u * h, qz = r.selz + 0x00020002u * h;
            // the exit planes are the entry planes of the swapped words
            nx[h] = __builtin_bit_cast(th2, __builtin_amdgcn_perm((uint32_t)I1.y, (uint32_t)I1.x, qx));
            fx[h] = __builtin_bit_cast(th2, __builtin_amdgcn_perm((uint32_t)I1.x, (uint32_t)I1.y, qx));
            ny[h] = __builtin_bit_cast(th2, __builtin_amdgcn_perm((uint32_t)I1.w, (uint32_t)I1.z, qy));
            fy[h] = __builtin_bit_cast(th2, __builtin_amdgcn_perm((uint32_t)I1.z, (uint32_t)I1.w, qy));
            nz[h] = __builtin_bit_cast(th2, __builtin_amdgcn_perm((uint32_t)I2.y, (uint32_t)I2.x, qz));
            fz[h] = __builtin_bit_cast(th2, __builtin_amdgcn_perm((uint32_t)I2.x, (uint32_t)I2.y, qz));
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
        {
            const int h = c >> 1, k = c & 1;
            const float x0 = __builtin_fmaf((float)nx[h][k], sx, bx), x1 = __builtin_fmaf((float)fx[h][k], sx, bx);
            const float y0 = __builtin_fmaf((float)ny[h][k], sy, by), y1 = __builtin_fmaf((float)fy[h][k], sy, by);
            const float z0 = __builtin_fmaf((float)nz[h][k], sz, bz), z1 = __builtin_fmaf((float)fz[h][k], sz, bz);
            tn[c] = fmaxf(fmaxf(x0, y0), fmaxf(z0, r.tmin));
            df[c] = fminf(fminf(x1, y1), fminf(z1, r.tcur)) - tn[c];
        }
    }
    else
    {
        const size_t nb = 8 * (size_t)node;
        const float4 LX = gload(nodes, nb), HX = gload(nodes, nb + 1), LY = gload(nodes, nb + 2),
                     HY = gload(nodes, nb + 3), LZ = gload(nodes, nb + 4), HZ = gload(nodes, nb + 5);
        const int4 REF = gload_i(nodes, nb + 6), CNT = gload_i(nodes, nb + 7);
        const float lx[4] = {LX.x, LX.y, LX.z, LX.w}, hx[4] = {HX.x, HX.y, HX.z, HX.w};
        const float ly[4] = {LY.x, LY.y, LY.z, LY.w}, hy[4] = {HY.x, HY.y, HY.z, HY.w};
        const float lz[4] = {LZ.x, LZ.y, LZ.z, LZ.w}, hz[4] = {HZ.x, HZ.y, HZ.z, HZ.w};
        const int cn[4] = {CNT.x, CNT.y, CNT.z, CNT.w};
        ref[0] = REF.x; ref[1] = REF.y; ref[2] = REF.z; ref[3] = REF.w;
        cnts = leaf = 0u;
#pragma unroll
        for (int c = 0; c < 4; ++c)
        {
            const float x0 = __builtin_fmaf(lx[c], r.ix, -r.ox), x1 = __builtin_fmaf(hx[c], r.ix, -r.ox);
            const float y0 = __builtin_fmaf(ly[c], r.iy, -r.oy), y1 = __builtin_fmaf(hy[c], r.iy, -r.oy);
            const float z0 = __builtin_fmaf(lz[c], r.iz, -r.oz), z1 = __builtin_fmaf(hz[c], r.iz, -r.oz);
            tn[c] = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fmaxf(fminf(z0, z1), r.tmin));
            df[c] = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fminf(fmaxf(z0, z1), r.tcur)) - tn[c];
            cnts |= ((uint32_t)cn[c] & 0xffu) << (8 * c);
            leaf |= cn[c] > 0 ? ((1u << cn[c]) - 1u) << (8 * c) : 0u;
        }
    }
    // byte c = 0xff where child c is missed (exit - entry negative: v_perm selectors 9 and 11
    // replicate the sign bit of the second and of the first source)
    const uint32_t miss = __builtin_amdgcn_perm(__float_as_uint(df[1]), __float_as_uint(df[0]), 0x0c0c0b09u) |
                          __builtin_amdgcn_perm(__float_as_uint(df[3]), __float_as_uint(df[2]), 0x0b090c0cu);
    r.base = (uint32_t)ref[0] - 1u;
    r.full = leaf;
    r.pend = leaf & ~miss;
    // key = the entry distance of a hit internal child, else a sentinel; a leaf's count is 1 to 8 and
    // an empty or missed child's byte 0xff
    const uint32_t out = miss | cnts;
    double key[4];
    if (kAnyMin)
    {
        // as v_perm selectors those bytes pick 0xff, and 0 picks 0
        uint32_t lut = 0xffffff00u, none = kKeyNone;
        asm("" : "+s"(lut), "+s"(none));   // in scalar registers, not moved or combined in vector ones
        const uint32_t skip = __builtin_amdgcn_perm(0xffffffffu, lut, out);
#pragma unroll
        for (int c = 0; c < 4; ++c)
        {
            const uint32_t m = __builtin_amdgcn_perm(skip, skip, 0x01010101u * (uint32_t)c);
            key[c] = key_pair(__uint_as_float((m & none) | (~m & __float_as_uint(tn[c]))), (uint32_t)ref[c]);
        }
    }
    else
    {
#pragma unroll
        for (int c = 0; c < 4; ++c)
            key[c] = key_pair(__builtin_fmaf((float)((out >> (8 * c)) & 0xffu), kKeyFar, tn[c]), (uint32_t)ref[c]);
    }
    r.k0 = key[0];
    r.k1 = key[1];
    r.k2 = key[2];
    r.k3 = key[3];
}

// The lane's stack: `top` in a register, the other entries in LDS ([entry][lane], kStride lanes),
// past kLds entries in the lane's overflow slots.
template <int kLds, int kStride, class Ovf>
__device__ __forceinline__ void stack_put(uint32_t* stk, const Ovf& ovf, uint32_t& spb, uint32_t v)
{
    constexpr uint32_t row = 4u * kStride;
    if (spb < kLds * row) *(lu32*)((__attribute__((address_space(3))) char*)stk + spb) = v;
    else if (spb < (uint32_t)kMaxStack4 * row) ovf.at((int)(spb / row) - kLds) = v;
    else return;   // the builder bounds the depth, so this never drops an entry
    spb += row;
}

// Starts a ray: the root on top of an otherwise empty stack, and no children, so its first step
// visits the root.
template <int kStride>
__device__ __forceinline__ void start_ray(LaneRay& r, uint32_t* stk, float4 a, float4 b)
{
    r.o = mk(a.x, a.y, a.z);
    r.d = mk(b.x, b.y, b.z);
    const float dx = fabsf(r.d.x) < 1e-20f ? copysignf(1e-20f, r.d.x) : r.d.x;
    const float dy = fabsf(r.d.y) < 1e-20f ? copysignf(1e-20f, r.d.y) : r.d.y;
    const float dz = fabsf(r.d.z) < 1e-20f ? copysignf(1e-20f, r.d.z) : r.d.z;
    r.ix = rcp_exact(dx);
    r.iy = rcp_exact(dy);
    r.iz = rcp_exact(dz);
    r.ox = r.o.x * r.ix;
    r.oy = r.o.y * r.iy;
    r.oz = r.o.z * r.iz;
    r.selx = r.ix >= 0.f ? kSelLo : kSelHi;
    r.sely = r.iy >= 0.f ? kSelLo : kSelHi;
    r.selz = r.iz >= 0.f ? kSelLo : kSelHi;
    r.tmin = a.w;
    r.tcur = b.w;
    r.prim = -1;
    r.b1 = r.b2 = 0.f;
    r.pend = 0u;
    r.k0 = r.k1 = r.k2 = r.k3 = key_pair(__builtin_inff(), 0u);
    r.top = 0u;
    r.spb = 4u * (threadIdx.x & (kStride - 1));
    *(lu32*)((__attribute__((address_space(3))) char*)stk + r.spb) = kStackEnd;
    r.spb += 4u * kStride;
}

// One step of an active lane: a pending leaf triangle, then, once the lane's leaves are done, its
// internal children (culled against the closest hit, nearest first) and the next node's visit.
// The order of box and triangle tests is traverse4's. Returns true when the ray is finished.
template <bool kCount, bool kQ, bool kOne, bool kAnyMin, int kLds, int kStride, class Ovf>
__device__ __forceinline__ bool step4(LaneRay& r, bool any, const float4* nodes, const float4* tris, uint32_t* stk,
                                      const Ovf& ovf, uint32_t& nvis, uint32_t& tvis)
{
    constexpr uint32_t row = 4u * kStride;
    typedef __attribute__((address_space(3))) char lchar;
    bool done = false;
    if (r.pend)
    {
        // the lowest pending bit is triangle (number of leaf bits below it) of the node's leaves
        const uint32_t m1 = r.pend - 1u;
        const uint32_t tq = r.base + (uint32_t)__popc(r.full & (r.pend ^ m1));
        r.pend &= m1;
        const float4* tp = kOne ? reinterpret_cast<const float4*>(reinterpret_cast<const char*>(tris) + tq * 48u)
                                : tris + 3 * (size_t)tq;
        const float4 v0 = gload(tp, 0), a1 = gload(tp, 1), a2 = gload(tp, 2);
        if (kCount) ++tvis;
        float t, u, v;
        if (intersect_face_dev(ld3(v0), ld3(a1), ld3(a2), r.o, r.d, r.tmin, r.tcur, t, u, v))
        {
            r.prim = __float_as_int(v0.w);
            r.tcur = t;
            r.b1 = u;
            r.b2 = v;
            done = any;
        }
    }
    if (!done && r.pend == 0u)
    {
        pair_sort2(r.k0, r.k1);
        pair_sort2(r.k2, r.k3);
        pair_sort2(r.k0, r.k2);
        pair_sort2(r.k1, r.k3);
        pair_sort2(r.k1, r.k2);
        // the children not beyond the closest hit are the first ones of the sorted four
        // (entered at +inf, a child is not visited in either form)
        const float tc = fminf(r.tcur, kAnyMin ? 3.4028235e38f : kKeyMost);
        const bool c0 = pair_key(r.k0) <= tc, c1 = pair_key(r.k1) <= tc, c2 = pair_key(r.k2) <= tc,
                   c3 = pair_key(r.k3) <= tc;
        uint32_t node = pair_id(r.k0);
        // one wave-uniform test instead of one per push: does any lane come near the LDS part's end
        const bool deep = __any(r.spb > (kLds - 3) * row + (row - 1u));
        if (!deep)
        {
            if (c1)
            {
                *(lu32*)((lchar*)stk + r.spb) = r.top;
                r.spb += row;
                if (c2)
                {
                    if (c3)
                    {
                        *(lu32*)((lchar*)stk + r.spb) = pair_id(r.k3);
                        r.spb += row;
                    }
                    *(lu32*)((lchar*)stk + r.spb) = pair_id(r.k2);
                    r.spb += row;
                }
                r.top = pair_id(r.k1);
            }
        }
        else if (c1)
        {
            stack_put<kLds, kStride>(stk, ovf, r.spb, r.top);
            if (c3) stack_put<kLds, kStride>(stk, ovf, r.spb, pair_id(r.k3));
            if (c2) stack_put<kLds, kStride>(stk, ovf, r.spb, pair_id(r.k2));
            r.top = pair_id(r.k1);
        }
        if (!c0)
        {
            node = r.top;
            if (node == kStackEnd) done = true;
            else
            {
                r.spb -= row;
                if (!deep || r.spb < kLds * row) r.top = *(lu32*)((lchar*)stk + r.spb);
                else r.top = ovf.at((int)(r.spb / row) - kLds);
            }
        }
        if (!done)
        {
            if (kCount) ++nvis;
            visit4<kQ, kOne, kAnyMin>(r, nodes, node);
        }
    }
    return done;
}

}  // namespace bsh
