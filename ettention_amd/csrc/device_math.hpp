// Device-side building blocks of the projectors: storage conversion, the DDA
// ray traversal and the fract of the bilinear lookups.  Every file including this
// is compiled with -ffp-contract=off: the expressions below round exactly as
// the OpenCL C source of the reference writes them, so the traversal takes
// the same voxel sequence and the same segment lengths.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>

#include "kernels.hpp"

namespace etn {
namespace dev {

constexpr float kEpsilon = 1e-4f;     // ocl_src/Math.hl:4

// Global-memory pointers.  A pointer read from a descriptor table in memory is
// a generic pointer to the compiler, and accesses through it become flat
// instructions (issued to both the memory and the LDS pipes, results in
// VGPRs); marking it global gives global loads and scalar loads of uniform data.
// (The host pass of the single-source compile only parses device code: no
// address space there.)
// Marking a table constant (it is not written while the kernel runs) turns
// its uniform reads into scalar loads even after the kernel's own stores:
// a vector load of a per-projection parameter would otherwise wait (vmcnt, in
// issue order) for every band load issued before it.
#ifdef __HIP_DEVICE_COMPILE__
#define ETN_GLOBAL __attribute__((address_space(1)))
#define ETN_CONST __attribute__((address_space(4)))
#else
#define ETN_GLOBAL
#define ETN_CONST
#endif
template <typename T>
__device__ __forceinline__ ETN_GLOBAL T* global_ptr(T* p)
{
    return (ETN_GLOBAL T*)p;
}
template <typename T>
__device__ __forceinline__ const ETN_CONST T* const_ptr(const ETN_GLOBAL T* p)
{
    return (const ETN_CONST T*)(const T*)p;
}

// ---- voxel storage ---------------------------------------------------------
// load/store take any pointer to T (generic or global)
// Stochastic rounding (opt-in for 16-bit storage): f goes to one of the two
// representable values enclosing it, "down" (toward zero) and "up", and to
// "up" with probability (f - down) / (up - down), so the stored value is f in
// expectation: updates smaller than half a unit in the last place survive on
// average instead of being dropped.  r holds uniformly distributed bits.
__device__ __forceinline__ uint32_t sr_hash(uint32_t index, uint32_t salt, float value)
{
    // murmur3's 32-bit finaliser over the voxel index, the projection's salt
    // and the value being rounded (which changes from one update to the next)
    uint32_t h = index * 0x9E3779B1u ^ salt * 0x85EBCA77u ^ __float_as_uint(value);
    h ^= h >> 16;
    h *= 0x85EBCA6Bu;
    h ^= h >> 13;
    h *= 0xC2B2AE35u;
    h ^= h >> 16;
    return h;
}

struct F32 {
    using T = float;
    template <typename P>
    static __device__ __forceinline__ float load(P p, size_t i) { return p[i]; }
    static __device__ __forceinline__ float round(float f) { return f; }
    static __device__ __forceinline__ float round_stochastic(float f, uint32_t) { return f; }
    template <typename P>
    static __device__ __forceinline__ void store(P p, size_t i, float f) { p[i] = f; }
};
struct F16 {   // vload_half / vstore_half (round to nearest even), HalfFloatSupport.hl:6-9
    using T = __half;
    template <typename P>
    static __device__ __forceinline__ float load(P p, size_t i)
    {
        const __half h = p[i];
        return __half2float(h);
    }
    static __device__ __forceinline__ float round(float f) { return __half2float(__float2half_rn(f)); }
    static __device__ __forceinline__ float round_stochastic(float f, uint32_t r)
    {
        // down: f rounded toward zero (exact when f is representable); up: the
        // next half away from zero (the sign kept; past the largest finite
        // half that is infinity, as round to nearest gives there too)
        const __half dn = __float2half_rz(f);
        const float d = __half2float(dn);
        const __half up = __ushort_as_half((unsigned short)(__half_as_ushort(dn) + 1u));
        const float u = __half2float(up);
        const float t = (float)(r >> 8) * 0x1.0p-24f;   // uniform in [0, 1)
        return fabsf(f - d) > t * fabsf(u - d) ? u : d;
    }
    template <typename P>
    static __device__ __forceinline__ void store(P p, size_t i, float f) { p[i] = __float2half_rn(f); }
    // two values in one v_cvt_pk_f16_f32 (gfx950, round to nearest even like
    // __float2half_rn): a in the low half, b in the high half
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ uint32_t pack2(float a, float b)
    {
        const f32x2 v = {a, b};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
    }
    // the two halves of a packed pair, low half first (exact)
    static __device__ __forceinline__ void unpack2(uint32_t h, float& a, float& b)
    {
        const f32x2 v = __builtin_convertvector(__builtin_bit_cast(f16x2, h), f32x2);
        a = v.x;
        b = v.y;
    }
};
struct BF16 {  // bfloat16, round to nearest even
    using T = uint16_t;
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    // two values in one v_cvt_pk_bf16_f32 (gfx950's conversion, round to
    // nearest even; a NaN stays a NaN): a in the low half, b in the high half
    static __device__ __forceinline__ uint32_t pack2(float a, float b)
    {
        const f32x2 v = {a, b};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
    }
    static __device__ __forceinline__ uint16_t pack(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
    static __device__ __forceinline__ float unpack(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
    static __device__ __forceinline__ void unpack2(uint32_t h, float& a, float& b)
    {
        a = __uint_as_float(h << 16);
        b = __uint_as_float(h & 0xffff0000u);
    }
    template <typename P>
    static __device__ __forceinline__ float load(P p, size_t i) { return unpack(p[i]); }
    static __device__ __forceinline__ float round(float f) { return unpack(pack(f)); }
    static __device__ __forceinline__ float round_stochastic(float f, uint32_t r)
    {
        // add 16 random bits below the kept mantissa and truncate: the
        // magnitude rounds up with probability equal to the dropped fraction
        const uint32_t u = __float_as_uint(f);
        if ((u & 0x7fffffffu) >= 0x7f800000u) return f;   // infinity, NaN
        return __uint_as_float((u + (r & 0xffffu)) & 0xffff0000u);
    }
    template <typename P>
    static __device__ __forceinline__ void store(P p, size_t i, float f) { p[i] = pack(f); }
};

// ---- DDA ray traversal (ocl_src/DDARaytracer.hl:20-110, RayUtils.hl:7-35) ---

// Per-projection constants of the traversal.
struct DdaConst {
    float ray[3], inv[3], step[3];
    int sign[3];
};

__device__ __forceinline__ DdaConst dda_const(const float ray[3], const float vs[3])
{
    DdaConst c;
    for (int k = 0; k < 3; ++k) {
        c.ray[k] = ray[k];
        // invertVectorSafely (RayUtils.hl:25-35)
        c.inv[k] = 1.0f / ray[k];
        if (ray[k] == 0.0f) c.inv[k] = -FLT_MAX;
        const float sg = ray[k] > 0.0f ? 1.0f : (ray[k] < 0.0f ? -1.0f : 0.0f);
        c.step[k] = vs[k] * c.inv[k] * sg;    // stepDifference = voxelSize * invRay * sign(ray)
        c.sign[k] = (int)sg;
    }
    return c;
}

// Traversal state of one ray.
struct DdaRay {
    int vox[3];
    float res[3];
    float acc, accl;
    uint32_t brk;
    int live;
};

// Entry into the subvolume box; leaves the ray dead when it misses
// (getBoundingBoxEntryAndExitPointInRayCoordinates, doesRayIntersectBoundingBox,
// calculateRayEntryPoint, getInitialVoxelIndex, getRemainingDifferenceToVoxelBorder).
__device__ __forceinline__ void dda_begin(const SlabParams& s, const DdaConst& c, const float src[3], DdaRay& r)
{
    float tmin[3], tmax[3];
    for (int k = 0; k < 3; ++k) {
        const float t0 = (s.bmin[k] - src[k]) * c.inv[k];
        const float t1 = (s.bmax[k] - src[k]) * c.inv[k];
        tmin[k] = fminf(t0, t1);
        tmax[k] = fmaxf(t0, t1);
    }
    const float t_in = fmaxf(fmaxf(tmin[0], tmin[1]), tmin[2]);
    const float t_out = fminf(fminf(tmax[0], tmax[1]), tmax[2]);
    r.acc = 0.0f;
    r.accl = 0.0f;
    r.brk = 0;
    r.live = (t_out - t_in > kEpsilon) ? 1 : 0;
    if (!r.live) {
        r.vox[0] = r.vox[1] = r.vox[2] = -1;
        r.res[0] = r.res[1] = r.res[2] = 0.0f;
        return;
    }
    for (int k = 0; k < 3; ++k) {
        const float ivs = 1.0f / s.vs[k];
        float p = src[k] + t_in * c.ray[k];
        p = fminf(fmaxf(p, s.bmin[k]), s.bmax[k]);
        int vi = (int)((p - s.bmin[k]) * ivs);      // convert_int4_rtz
        vi = max(vi, 0);
        vi = min(vi, s.res[k] - 1);
        r.vox[k] = vi;
        float d = floorf(p * ivs) * s.vs[k];
        d = (c.ray[k] > 0.0f) ? (d + s.vs[k] - p) * c.inv[k] : (d - p) * c.inv[k];
        d = (c.ray[k] == 0.0f) ? FLT_MAX : d;
        d = (d == 0.0f) ? c.step[k] : d;
        r.res[k] = d;
    }
}

// Sub-ray origin (ParallelBeamsForwardProjection.cl:12-24).
__device__ __forceinline__ void fp_ray_source(const RayParams& g, uint32_t x, uint32_t y, uint32_t si, uint32_t sj,
                                              float sd, float off, float src[3])
{
    const float fx = (float)x + off + sd * (float)si;
    const float fy = (float)y + off + sd * (float)sj;
    for (int k = 0; k < 3; ++k) {
        const float ru = g.h[k] * fx;
        const float rv = g.v[k] * fy;
        src[k] = g.source[k] + ru + rv;
    }
}

// ---- fract of the bilinear lookups (ocl_src/ImageHandler.hl:20-29) ----------
__device__ __forceinline__ float cl_fract(float x, float* base)
{
    const float fl = floorf(x);
    *base = fl;
    return fminf(x - fl, 0x1.fffffep-1f);
}

}  // namespace dev
}  // namespace etn
