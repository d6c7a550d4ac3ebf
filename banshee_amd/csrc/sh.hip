// Spherical-harmonic kernels: environment-map projection (ShProjectEnvironmentMap,
// math/shproject.cpp:73-130), irradiance from SH (ShTracer::GetE, tracer/shtracer.cpp:20-36)
// and the basis diagnostic. Probe baking lives with the wavefront kernels in render.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>
#include <vector>

#include "env_tiles.h"
#include "internal.h"
#include "sh_dev.h"

namespace bsh {

// The context's scratch for it: twice the 150 KB that kEnvMaxBlocks blocks' sums take at lmax 4, since
// maps of many columns or rows need more blocks.
constexpr size_t kEnvCtxFloats = (size_t)2 * kEnvMaxBlocks * 3 * kShMaxTerms;

// Environment projection: c_i = sum over the map's cells of e Y_i(w) sin(theta) (pi / H) (2 pi / W).
// Pass 1: a block takes a tile of kShTile columns (phi; the columns of a narrower map in several
// rows at a time) and `rows` rows (theta); each thread keeps its column and sums its rows' terms in
// registers, then the block adds its threads' sums in LDS, one channel at a time, in a fixed order.
// Bound by the map's 12 B per cell, then by the basis (about 60 instructions per cell at lmax 2).
// Lanes read consecutive texels (the loop order of the reference, theta inner, put them a map row
// apart), and the block reduces once per coefficient and 256 threads, not with eight barriers per
// coefficient and 256 cells: 2048 x 1024, lmax 2: 88 -> 13 us, and pass 2, whose one block walked
// 8192 partial sums per coefficient, 1634 -> 4 us; the call, which also filled its angle tables on
// the host and allocated, with 262,144 irradiances 1773 -> 33 us.
template <int LMAX>
__global__ __launch_bounds__(kShBlock) void k_env_partial(const float* __restrict__ env, int W, int H, EnvTiles tiles,
                                                        float* __restrict__ partial)
{
    constexpr int NT = (LMAX + 1) * (LMAX + 1);
    constexpr int kPitch = kShBlock + 1;
    __shared__ float red[NT * kPitch];
    __shared__ float s_sin[kShBlock], s_cos[kShBlock], s_w[kShBlock];
    const int t = threadIdx.x;
    // the angles in float as the reference forms them (shproject.cpp:85-104), their sines and
    // cosines rounded from double
    const float thetastep = kPi / H, phistep = 2.f * kPi / W;
    const float theta0 = kPi / H / 2, phi0 = 2.f * kPi / W / 2;
    const int cols = tiles.cols;
    const EnvTile tile = env_tile(blockIdx.x, tiles, H);
    const int row0 = tile.row0, nrows = tile.row1 - row0;
    if (t < nrows)
    {
        const double a = (double)(theta0 + (float)(row0 + t) * thetastep);
        s_sin[t] = (float)sin(a);
        s_cos[t] = (float)cos(a);
        s_w[t] = s_sin[t] * thetastep * phistep;
    }
    __syncthreads();
    const int phi = tile.col0 + t % cols, sub = t / cols, nsub = kShBlock / cols;
    float c[3 * NT];
#pragma unroll
    for (int i = 0; i < 3 * NT; ++i) c[i] = 0.f;
    if (phi < W && sub < nsub)
    {
        const double a = (double)(phi0 + (float)phi * phistep);
        const float sp = (float)sin(a), cp = (float)cos(a);
        // (from 2^24 columns or rows on the quotient may round up to 1, past the last texel)
        const int iu = min((int)floorf((float)phi / W * W), W - 1);
#pragma unroll 4
        for (int k = sub; k < nrows; k += nsub)
        {
            const int iv = min((int)floorf((float)(row0 + k) / H * H), H - 1);
            const float* e = env + 3 * ((size_t)W * iv + iu);
            const float st = s_sin[k], ct = s_cos[k], w = s_w[k];
            const float ex = e[0] * w, ey = e[1] * w, ez = e[2] * w;
            float y[NT];
            sh_poly<LMAX>(st * cp, ct, st * sp, y);
#pragma unroll
            for (int i = 0; i < NT; ++i)
            {
                c[3 * i + 0] = __builtin_fmaf(ex, y[i], c[3 * i + 0]);
                c[3 * i + 1] = __builtin_fmaf(ey, y[i], c[3 * i + 1]);
                c[3 * i + 2] = __builtin_fmaf(ez, y[i], c[3 * i + 2]);
            }
        }
    }
    const int nblocks = gridDim.x, block = blockIdx.x;
#pragma unroll
    for (int ch = 0; ch < 3; ++ch)
    {
#pragma unroll
        for (int i = 0; i < NT; ++i) red[i * kPitch + t] = c[3 * i + ch];
        __syncthreads();
        // 8 threads per coefficient add 32 sums each, then one another's
        for (int i = t >> 3; i < NT; i += kShBlock / 8)
        {
            float s = 0.f;
#pragma unroll 8
            for (int k = 0; k < kShBlock / 8; ++k) s += red[i * kPitch + 8 * k + (t & 7)];
            s += __shfl_xor(s, 1);
            s += __shfl_xor(s, 2);
            s += __shfl_xor(s, 4);
            if ((t & 7) == 0) partial[(size_t)(3 * i + ch) * nblocks + block] = s;
        }
        __syncthreads();
    }
}

// Pass 2: one wave per coefficient and channel adds the blocks' sums in a fixed order.
__global__ __launch_bounds__(64) void k_env_final(const float* __restrict__ partial, int nblocks, float* coeffs)
{
    const float* p = partial + (size_t)blockIdx.x * nblocks;
    float s = 0.f;
    for (int b = threadIdx.x; b < nblocks; b += 64) s += p[b];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off);
    if (threadIdx.x == 0) coeffs[blockIdx.x] = s;
}

// lmax as a template argument: the basis stays in registers and its constants are folded (with lmax
// at run time 262,144 normals took 9.5 us, now 4.1); the operations and their order are the same.
template <int LMAX>
__global__ __launch_bounds__(256) void k_irradiance(const float* __restrict__ coeffs, const float* __restrict__ normals,
                                                    uint32_t n, float* __restrict__ out)
{
    uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    float y[kShMaxTerms];
    sh_evaluate(mk(normals[3 * (size_t)t], normals[3 * (size_t)t + 1], normals[3 * (size_t)t + 2]), LMAX, y);
    f3 e = mk(0.f, 0.f, 0.f);
#pragma unroll
    for (int l = 0; l <= LMAX; ++l)
    {
        float lam = sh_lambda(l);
#pragma unroll
        for (int m = -l; m <= l; ++m)
        {
            int o = sh_index(l, m);
            // ShConvolveCosTheta: lambda(l) * cin * s_costheta[l]
            f3 cc = lam * mk(coeffs[3 * o], coeffs[3 * o + 1], coeffs[3 * o + 2]) * sh_costheta(l);
            e = e + y[o] * cc * (0.7f / 3.14159265358979323846f);
        }
    }
    out[3 * (size_t)t] = e.x;
    out[3 * (size_t)t + 1] = e.y;
    out[3 * (size_t)t + 2] = e.z;
}

__global__ void k_diag_sh(int lmax, uint32_t n, const float* dirs, float* out)
{
    uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    int nt = (lmax + 1) * (lmax + 1);
    float y[kShMaxTerms];
    sh_evaluate(mk(dirs[3 * t], dirs[3 * t + 1], dirs[3 * t + 2]), lmax, y);
    for (int i = 0; i < nt; ++i) out[(size_t)t * nt + i] = y[i];
}

static size_t env_partial_floats(int W, int H, int lmax)
{
    const EnvTiles t = env_tiles(W, H);
    return (size_t)t.nx * t.ny * 3 * (lmax + 1) * (lmax + 1);
}

static bsh_status check_env_args(bsh_context* ctx, const float* env, int width, int height, int lmax,
                                 const float* coeffs, const char* who)
{
    std::string w(who);
    if (!ctx || !env || !coeffs) return fail(BSH_ERR_INVALID, w + ": NULL argument");
    if (width <= 0 || height <= 0) return fail(BSH_ERR_INVALID, w + ": bad size");
    if (lmax < 0 || lmax > kShMaxL) return fail(BSH_ERR_UNSUPPORTED, w + ": lmax must be 0..4");
    if ((size_t)width * height >= ((size_t)1 << 31)) return fail(BSH_ERR_UNSUPPORTED, w + ": too large");
    return BSH_OK;
}

// Both passes; `partial` holds env_partial_floats(W, H, lmax) floats, every one written by pass 1.
static hipError_t launch_env_projection(const float* env, int W, int H, int lmax, float* partial, float* coeffs,
                                        hipStream_t st)
{
    const EnvTiles q = env_tiles(W, H);
    const dim3 g((uint32_t)(q.nx * q.ny)), b(kShBlock);
    switch (lmax)
    {
    case 0: hipLaunchKernelGGL(k_env_partial<0>, g, b, 0, st, env, W, H, q, partial); break;
    case 1: hipLaunchKernelGGL(k_env_partial<1>, g, b, 0, st, env, W, H, q, partial); break;
    case 2: hipLaunchKernelGGL(k_env_partial<2>, g, b, 0, st, env, W, H, q, partial); break;
    case 3: hipLaunchKernelGGL(k_env_partial<3>, g, b, 0, st, env, W, H, q, partial); break;
    default: hipLaunchKernelGGL(k_env_partial<4>, g, b, 0, st, env, W, H, q, partial); break;
    }
    hipLaunchKernelGGL(k_env_final, dim3(3 * (lmax + 1) * (lmax + 1)), dim3(64), 0, st, (const float*)partial,
                       q.nx * q.ny, coeffs);
    return hipGetLastError();
}

// Scratch of the allocation-free projection: one copy per device, held until the process
// ends. Calls on one device share it, so calls that overlap on one device race.
static __device__ __align__(256) float scratch[kEnvScratchFloats];

static std::mutex g_scratch_mu;
static float* g_scratch_dev[kMaxDevices] = {};

// Device address of `scratch` on `device`, looked up once per device with that device
// current (in host code the array's name is only a stand-in for it).
bsh_status env_scratch_init(int device)
{
    if (device < 0 || device >= kMaxDevices) return fail(BSH_ERR_UNSUPPORTED, "device index beyond the scratch table");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_dev[device]) return BSH_OK;
    BSH_HIP(hipSetDevice(device));
    void* p = nullptr;
    BSH_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return fail(BSH_ERR_STATE, "hipGetSymbolAddress(scratch) returned NULL");
    g_scratch_dev[device] = (float*)p;
    return BSH_OK;
}

float* env_scratch_ptr(int device)
{
    if (device < 0 || device >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    return g_scratch_dev[device];
}

}  // namespace bsh

using namespace bsh;

extern "C" {

bsh_status bsh_sh_project_env(bsh_context* ctx, const float* env, int width, int height, int lmax, float* coeffs,
                              void* stream)
{
    bsh_status v = check_env_args(ctx, env, width, height, lmax, coeffs, "bsh_sh_project_env");
    if (v != BSH_OK) return v;
    BSH_HIP(hipSetDevice(ctx->device));
    hipStream_t st = (hipStream_t)stream;
    // the context's scratch while no other call is using it, else (another thread's call is in
    // flight, or the map has more blocks than the scratch holds) an allocation of this call's own
    const size_t need = env_partial_floats(width, height, lmax);
    std::unique_lock<std::mutex> lk(ctx->env_mu, std::try_to_lock);
    DevBuf<float> own;
    float* part = nullptr;
    if (lk.owns_lock() && need <= kEnvCtxFloats)
    {
        BSH_HIP(ctx->env_part.alloc(kEnvCtxFloats));
        part = ctx->env_part.p;
    }
    else
    {
        BSH_HIP(own.alloc(need));
        part = own.p;
    }
    BSH_HIP(launch_env_projection(env, width, height, lmax, part, coeffs, st));
    BSH_HIP(hipStreamSynchronize(st));   // the sums are read before the scratch is given back
    return BSH_OK;
}

bsh_status bsh_sh_project_env_noalloc(bsh_context* ctx, const float* env, int width, int height, int lmax,
                                      float* coeffs, void* stream)
{
    bsh_status v = check_env_args(ctx, env, width, height, lmax, coeffs, "bsh_sh_project_env_noalloc");
    if (v != BSH_OK) return v;
    // the documented limit: two tables of a map's angles and 3 (lmax + 1)^2 sums per 256 cells
    const size_t ntab = 2 * ((size_t)width + height);
    const size_t npart = ((size_t)width * height + 255) / 256 * 3 * (lmax + 1) * (lmax + 1);
    const size_t part_off = (ntab + 63) & ~(size_t)63;
    if (part_off + npart > kEnvScratchFloats || env_partial_floats(width, height, lmax) > kEnvScratchFloats)
        return fail(BSH_ERR_INVALID, "bsh_sh_project_env_noalloc: a " + std::to_string(width) + "x" +
                                         std::to_string(height) + " map at lmax " + std::to_string(lmax) + " needs " +
                                         std::to_string((part_off + npart) * 4) + " B of scratch, more than its " +
                                         std::to_string(kEnvScratchFloats * 4) + " B; use bsh_sh_project_env");
    BSH_HIP(hipSetDevice(ctx->device));
    float* base = env_scratch_ptr(ctx->device);
    if (!base) return fail(BSH_ERR_STATE, "bsh_sh_project_env_noalloc: scratch of device " +
                                              std::to_string(ctx->device) + " was not set up by bsh_context_create");
    hipStream_t st = (hipStream_t)stream;
    BSH_HIP(launch_env_projection(env, width, height, lmax, base, coeffs, st));
    return BSH_OK;
}

bsh_status bsh_sh_irradiance(bsh_context* ctx, int lmax, const float* coeffs, const float* normals, size_t n,
                             float* out, void* stream)
{
    if (!ctx || !coeffs || (n && (!normals || !out))) return fail(BSH_ERR_INVALID, "bsh_sh_irradiance: NULL argument");
    if (lmax < 0 || lmax > kShMaxL) return fail(BSH_ERR_UNSUPPORTED, "bsh_sh_irradiance: lmax must be 0..4");
    if (n == 0) return BSH_OK;
    BSH_HIP(hipSetDevice(ctx->device));
    const dim3 g((uint32_t)((n + 255) / 256)), b(256);
    switch (lmax)
    {
    case 0: hipLaunchKernelGGL(k_irradiance<0>, g, b, 0, (hipStream_t)stream, coeffs, normals, (uint32_t)n, out); break;
    case 1: hipLaunchKernelGGL(k_irradiance<1>, g, b, 0, (hipStream_t)stream, coeffs, normals, (uint32_t)n, out); break;
    case 2: hipLaunchKernelGGL(k_irradiance<2>, g, b, 0, (hipStream_t)stream, coeffs, normals, (uint32_t)n, out); break;
    case 3: hipLaunchKernelGGL(k_irradiance<3>, g, b, 0, (hipStream_t)stream, coeffs, normals, (uint32_t)n, out); break;
    default: hipLaunchKernelGGL(k_irradiance<4>, g, b, 0, (hipStream_t)stream, coeffs, normals, (uint32_t)n, out); break;
    }
    BSH_HIP(hipGetLastError());
    return BSH_OK;
}

bsh_status bsh_diag_sh_eval(bsh_context* ctx, int lmax, size_t n, const float* dirs, float* out)
{
    if (!ctx || (n && (!dirs || !out))) return fail(BSH_ERR_INVALID, "bsh_diag_sh_eval: NULL argument");
    if (lmax < 0 || lmax > kShMaxL) return fail(BSH_ERR_UNSUPPORTED, "bsh_diag_sh_eval: lmax must be 0..4");
    if (n == 0) return BSH_OK;
    BSH_HIP(hipSetDevice(ctx->device));
    int nt = (lmax + 1) * (lmax + 1);
    DevBuf<float> d, o;
    BSH_HIP(d.alloc(3 * n));
    BSH_HIP(o.alloc(nt * n));
    BSH_HIP(hipMemcpy(d.p, dirs, 3 * n * 4, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_diag_sh, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, 0, lmax, (uint32_t)n, d.p, o.p);
    BSH_HIP(hipGetLastError());
    BSH_HIP(hipMemcpy(out, o.p, nt * n * 4, hipMemcpyDeviceToHost));
    return BSH_OK;
}

}  // extern "C"
