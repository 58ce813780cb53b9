// Generic gfx950 kernels of the SART hot path: one thread per detector pixel
// (forward projection, residual, long-object compensation, ray length) or per
// voxel (back projection), for any parallel geometry, any subvolume split and
// any sample count.  The fused plane kernels (fused.hip) take over the common
// single-axis case; these serve everything else and the per-kernel C ABI.
#include <mutex>
#include <vector>

#include "device_math.hpp"
#include "common.hpp"

namespace etn {
namespace dev {

namespace {

// Mask weights of the 256 mask bytes (MaskVolume's byte / 255, ImageHandler.hl:
// 85-89), divided once per workgroup instead of once per voxel visited.
__device__ __forceinline__ void fill_mask_weights(float* weights)
{
    const int t = threadIdx.x + threadIdx.y * blockDim.x;
    if (t < 256) weights[t] = (float)t / 255.0f;
    __syncthreads();
}

// ParallelBeamsForwardProjection.cl:execute.  A pixel's sub-rays are spread over
// kSubs lanes (a power of two, as many as there are sub-rays up to 16) and their
// sums added in the reference's (si, sj) order.  A ray's voxels and segment
// lengths do not depend on what the voxels hold, so it takes kBatch steps ahead
// and reads their voxels together; the reference's loop, one dependent gather a
// step on too few waves to cover its latency, took 0.85 ms on 301 x 203 x 257
// with 2 x 2 sub-rays and a mask in f16 (0.29 ms).
constexpr int kFpBatch = 8;

template <typename S, bool kMask, int kSubs>
__global__ void __launch_bounds__(256) forward_project_kernel(SlabParams s, RayParams g, const typename S::T* vol,
                                                              const uint8_t* mask, float* proj, float* len)
{
    __shared__ float weights[kMask ? 256 : 1];
    if (kMask) fill_mask_weights(weights);
    const uint32_t sub = threadIdx.x % kSubs;
    const uint32_t x = (blockIdx.x * blockDim.x + threadIdx.x) / kSubs;
    const uint32_t y = blockIdx.y * blockDim.y + threadIdx.y;
    const bool pixel = x < g.nu && y < g.nv;
    const DdaConst c = dda_const(g.ray, s.vs);
    const uint32_t n = g.samples, count = n * n;
    const float total = (float)(n * n);
    const float sd = 1.0f / (float)n, off = sd / 2.0f;
    vol += s.first_voxel;
    if (kMask) mask += s.first_voxel;
    const ptrdiff_t step_y = (ptrdiff_t)c.sign[1] * (ptrdiff_t)s.nx, step_z = (ptrdiff_t)c.sign[2] * (ptrdiff_t)s.nx * s.ny;
    float acc = 0.0f, accl = 0.0f;
    for (uint32_t first = 0; first < count; first += kSubs) {
        const uint32_t k = first + sub;
        DdaRay r;
        r.acc = r.accl = 0.0f;
        if (pixel && k < count) {
            float src[3];
            fp_ray_source(g, x, y, k / n, k % n, sd, off, src);
            dda_begin(s, c, src, r);
            // the reference's loop condition (voxel in range, then ++breakVar < 4096,
            // with a second ++breakVar in the body: at most 2048 steps,
            // DDARaytracer.hl:20-110) as the steps left on each axis until the ray
            // leaves the volume, and in all
            uint32_t left = r.live ? 2048u : 0u;
            int lx = c.sign[0] > 0 ? s.res[0] - r.vox[0] : c.sign[0] < 0 ? r.vox[0] + 1 : 0x7fffffff;
            int ly = c.sign[1] > 0 ? s.res[1] - r.vox[1] : c.sign[1] < 0 ? r.vox[1] + 1 : 0x7fffffff;
            int lz = c.sign[2] > 0 ? s.res[2] - r.vox[2] : c.sign[2] < 0 ? r.vox[2] + 1 : 0x7fffffff;
            ptrdiff_t at = r.live ? ((ptrdiff_t)r.vox[2] * s.ny + r.vox[1]) * s.nx + r.vox[0] : 0;
            float rx = r.res[0], ry = r.res[1], rz = r.res[2];
            while (left != 0) {
                ptrdiff_t voxel[kFpBatch];
                float dt[kFpBatch];
                uint32_t steps = 0;
#pragma unroll
                for (int b = 0; b < kFpBatch; ++b) {
                    // (steps past the ray's end read its last voxel and add nothing)
                    voxel[b] = at;
                    dt[b] = fminf(fminf(rx, ry), rz);
                    if (left != 0) {
                        const bool ix = rx <= ry && rx <= rz, iy = ry < rx && ry <= rz, iz = rz < rx && rz < ry;
                        rx = ix ? c.step[0] : rx - dt[b];
                        ry = iy ? c.step[1] : ry - dt[b];
                        rz = iz ? c.step[2] : rz - dt[b];
                        lx -= ix ? 1 : 0;
                        ly -= iy ? 1 : 0;
                        lz -= iz ? 1 : 0;
                        left = lx != 0 && ly != 0 && lz != 0 ? left - 1 : 0;
                        ++steps;
                        // (the voxel after the last is not in the volume)
                        if (left != 0) at += ix ? (ptrdiff_t)c.sign[0] : iy ? step_y : iz ? step_z : 0;
                    }
                }
                float value[kFpBatch], maskv[kFpBatch];
#pragma unroll
                for (int b = 0; b < kFpBatch; ++b) {
                    value[b] = S::load(vol, (size_t)voxel[b]);
                    maskv[b] = kMask ? weights[mask[voxel[b]]] : 1.0f;
                }
#pragma unroll
                for (int b = 0; b < kFpBatch; ++b) {
                    if ((uint32_t)b < steps) {
                        r.acc += dt[b] * value[b];
                        r.accl += dt[b] * maskv[b];
                    }
                }
            }
        }
        if constexpr (kSubs == 1) {
            acc += r.acc;
            accl += r.accl;
        } else {
#pragma unroll
            for (int q = 0; q < kSubs; ++q) {
                const float a = __shfl(r.acc, q, kSubs), l = __shfl(r.accl, q, kSubs);
                if (first + q < count) {
                    acc += a;
                    accl += l;
                }
            }
        }
    }
    if (!pixel || sub != 0) return;
    const size_t i = (size_t)y * g.nu + x;
    proj[i] += acc / total;
    len[i] += accl / total;
}

// ParallelBeamsBackProjection.cl:correct for kBpDepth voxels of a column (its
// sample loop, :26-44: a sample with a ray length up to 1e-4 is not used): the
// x and y terms of the projected point serve all of them, and their image reads
// are in flight together.  kUnit: the matrix's last row is (0, 0, 0, 1), so that
// u and v are divided by exactly 1.  Residual and ray length are looked up at
// one place: one set of indices and weights for both.  301 x 203 x 257 in bf16
// with 4 samples and a mask: 0.23 -> 0.15 ms.
constexpr int kBpDepth = 4;

template <typename S, bool kMask, bool kUnit>
__global__ void __launch_bounds__(256) back_project_kernel(SlabParams s, BpParams b, typename S::T* vol,
                                                           const uint8_t* mask, const float* residual,
                                                           const float* ray_length)
{
    __shared__ float weights[kMask ? 256 : 1];
    if (kMask) fill_mask_weights(weights);
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    const int z0 = blockIdx.z * kBpDepth;
    if (x >= s.res[0] || y >= s.res[1]) return;
    const int nu = (int)b.nu, nv = (int)b.nv;
    const size_t slice = (size_t)s.ny * s.nx;
    const size_t i0 = s.first_voxel + (size_t)z0 * slice + (size_t)y * s.nx + (size_t)x;
    const float cx = s.bmin[0] + ((float)x + 0.5f) * s.vs[0], cy = s.bmin[1] + ((float)y + 0.5f) * s.vs[1];
    float value[kBpDepth], sum[kBpDepth], cz[kBpDepth];
    uint32_t used[kBpDepth];
#pragma unroll
    for (int d = 0; d < kBpDepth; ++d) {
        value[d] = z0 + d < s.res[2] ? S::load(vol, i0 + d * slice) : 0.0f;
        cz[d] = s.bmin[2] + ((float)(z0 + d) + 0.5f) * s.vs[2];
        sum[d] = 0.0f;
        used[d] = 0;
    }
    for (uint32_t si = 0; si < b.nsamples; ++si) {
        const float4 smp = b.samples[si];
        const float px = cx + smp.x, py = cy + smp.y;
        // detector coordinates (TransformCoordG, Matrix4x4.hl:38-58): the x and y
        // terms of the rows first
        const float ux = b.m[0] * px + b.m[4] * py, vx = b.m[1] * px + b.m[5] * py, wx = b.m[3] * px + b.m[7] * py;
#pragma unroll
        for (int d = 0; d < kBpDepth; ++d) {
            const float pz = cz[d] + smp.z;
            float u = ux + b.m[8] * pz, v = vx + b.m[9] * pz;
            u = u + b.m[12] * 1.0f;
            v = v + b.m[13] * 1.0f;
            if constexpr (!kUnit) {
                float w = wx + b.m[11] * pz;
                w = w + b.m[15] * 1.0f;
                u = u / w;
                v = v / w;
            }
            // bilinear lookups with a zero border in both images (ImageHandler.hl:20-40)
            float bu, bv;
            const float tx = cl_fract(u - 0.5f, &bu), ty = cl_fract(v - 0.5f, &bv);
            const int i = (int)bu, j = (int)bv;
            const bool c0 = i >= 0 && i < nu, c1 = i + 1 >= 0 && i + 1 < nu;
            const bool r0 = j >= 0 && j < nv, r1 = j + 1 >= 0 && j + 1 < nv;
            const uint32_t a0 = (uint32_t)min(max(j, 0), nv - 1) * (uint32_t)nu, a1 = (uint32_t)min(max(j + 1, 0), nv - 1) * (uint32_t)nu;
            const uint32_t k0 = (uint32_t)min(max(i, 0), nu - 1), k1 = (uint32_t)min(max(i + 1, 0), nu - 1);
            const float l00 = ray_length[a0 + k0], l01 = ray_length[a0 + k1], l10 = ray_length[a1 + k0], l11 = ray_length[a1 + k1];
            const float q00 = residual[a0 + k0], q01 = residual[a0 + k1], q10 = residual[a1 + k0], q11 = residual[a1 + k1];
            auto lookup = [&](float p00, float p01, float p10, float p11) {
                const float h0 = c0 ? p00 : 0.0f, h1 = c1 ? p01 : 0.0f, g0 = c0 ? p10 : 0.0f, g1 = c1 ? p11 : 0.0f;
                const float v0 = r0 ? h0 + (h1 - h0) * tx : 0.0f, v1 = r1 ? g0 + (g1 - g0) * tx : 0.0f;
                return v0 + (v1 - v0) * ty;
            };
            const float L = lookup(l00, l01, l10, l11);
            const float R = lookup(q00, q01, q10, q11);
            const float w = smp.w / L;
            const float contrib = R * b.lambda * w;
            sum[d] += (L > kEpsilon) ? contrib : 0.0f;
            used[d] += (L > kEpsilon) ? 1u : 0u;
        }
    }
#pragma unroll
    for (int d = 0; d < kBpDepth; ++d) {
        if (z0 + d >= s.res[2]) break;
        const size_t i = i0 + d * slice;
        if (used[d] != 0) {
            const float maskv = kMask ? weights[mask[i]] : 1.0f;
            value[d] += maskv * sum[d] / (float)used[d];
        }
        S::store(vol, i, value[d]);
    }
}

// the measured projection in its storage type (f32, or f16/bf16 stored projections)
template <typename S>
__global__ void compare_kernel(uint32_t n, const typename S::T* real, const float* virt, float* res)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) res[i] = S::load(real, i) - virt[i];
}

__global__ void loc_kernel(uint32_t n, float* proj, float* len, float c)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float l = len[i];
    proj[i] = l > kEpsilon ? proj[i] * c / l : 0.0f;
    len[i] = c;
}

// ComputeRayLength.cl:execute for pixel (x, y)
__device__ __forceinline__ float ray_length_at(const RayParams& g, const float bmin[3], const float bmax[3],
                                               uint32_t x, uint32_t y)
{
    float src[3];
    const float fx = ((float)x) + 0.5f, fy = ((float)y) + 0.5f;
    float tmin[3], tmax[3];
    for (int k = 0; k < 3; ++k) {
        const float ru = g.h[k] * fx, rv = g.v[k] * fy;
        src[k] = g.source[k] + ru + rv;
        float inv = 1.0f / g.ray[k];
        if (g.ray[k] == 0.0f) inv = -FLT_MAX;
        const float t0 = (bmin[k] - src[k]) * inv, t1 = (bmax[k] - src[k]) * inv;
        tmin[k] = fminf(t0, t1);
        tmax[k] = fmaxf(t0, t1);
    }
    const float t_in = fmaxf(fmaxf(tmin[0], tmin[1]), tmin[2]);
    const float t_out = fminf(fminf(tmax[0], tmax[1]), tmax[2]);
    return fmaxf(t_out - t_in, 0.0f);
}

__global__ void ray_length_kernel(RayParams g, float bx0, float by0, float bz0, float bx1, float by1, float bz1,
                                  float* out)
{
    const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t y = blockIdx.y * blockDim.y + threadIdx.y;
    if (x >= g.nu || y >= g.nv) return;
    const float bmin[3] = {bx0, by0, bz0}, bmax[3] = {bx1, by1, bz1};
    out[(size_t)y * g.nu + x] = ray_length_at(g, bmin, bmax, x, y);
}

// Image blockIdx.z of a batch: its geometry from gs, its lengths at out + z * stride.
__global__ void ray_length_batch_kernel(const RayParams* __restrict__ gs, float bx0, float by0, float bz0, float bx1,
                                        float by1, float bz1, float* out, size_t stride)
{
    const RayParams g = gs[blockIdx.z];
    const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t y = blockIdx.y * blockDim.y + threadIdx.y;
    if (x >= g.nu || y >= g.nv) return;
    const float bmin[3] = {bx0, by0, bz0}, bmax[3] = {bx1, by1, bz1};
    out[(size_t)blockIdx.z * stride + (size_t)y * g.nu + x] = ray_length_at(g, bmin, bmax, x, y);
}

// FP64 sum of squared differences: per-block partials, then one block sums
// the partials in a fixed order (deterministic).
constexpr int kSsdThreads = 256;
template <typename S>
__global__ void __launch_bounds__(kSsdThreads) ssd_partial_kernel(const typename S::T* a, const float* b, size_t n,
                                                                  double* partials)
{
    __shared__ double red[kSsdThreads];
    double acc = 0.0;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const double d = (double)S::load(a, i) - (b ? (double)b[i] : 0.0);
        acc += d * d;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = kSsdThreads / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = red[0];
}
__global__ void __launch_bounds__(kSsdThreads) ssd_final_kernel(const double* partials, uint32_t n, double* out)
{
    __shared__ double red[kSsdThreads];
    double acc = 0.0;
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) acc += partials[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = kSsdThreads / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] += red[0];
}

template <typename SS, typename DS>
__global__ void convert_kernel(const typename SS::T* src, typename DS::T* dst, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        DS::store(dst, i, SS::load(src, i));
}

template <typename S>
__global__ void fill_kernel(typename S::T* dst, float value, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        S::store(dst, i, value);
}

uint32_t grid_for(size_t n, uint32_t threads)
{
    const size_t blocks = (n + threads - 1) / threads;
    return (uint32_t)(blocks < 8192 ? (blocks ? blocks : 1) : 8192);
}

void check_launch(const char* what)
{
    hip_check(hipGetLastError(), what);
}

}  // namespace

namespace {

template <typename S, bool kMask>
void forward_project_typed(const SlabParams& s, const RayParams& r, const void* volume, const uint8_t* mask,
                           float* projection, float* traversal_length, hipStream_t stream)
{
    const auto* vol = static_cast<const typename S::T*>(volume);
    const uint32_t subs = r.samples * r.samples;
    auto launch = [&](auto kernel, uint32_t lanes) {
        const dim3 block(64, 4);
        const dim3 grid((r.nu * lanes + 63) / 64, (r.nv + 3) / 4);
        kernel<<<grid, block, 0, stream>>>(s, r, vol, mask, projection, traversal_length);
    };
    // as many lanes a pixel as it has sub-rays, to 16
    if (subs >= 16) launch(forward_project_kernel<S, kMask, 16>, 16);
    else if (subs >= 8) launch(forward_project_kernel<S, kMask, 8>, 8);
    else if (subs >= 4) launch(forward_project_kernel<S, kMask, 4>, 4);
    else launch(forward_project_kernel<S, kMask, 1>, 1);
}

template <typename S, bool kMask>
void back_project_typed(const SlabParams& s, const BpParams& b, void* volume, const uint8_t* mask,
                        const float* residual, const float* ray_length, hipStream_t stream)
{
    auto* vol = static_cast<typename S::T*>(volume);
    const dim3 block(64, 4);
    const dim3 grid((s.res[0] + 63) / 64, (s.res[1] + 3) / 4, (s.res[2] + kBpDepth - 1) / kBpDepth);
    // w = 0 x + 0 y + 0 z + 1 is exactly 1
    const bool unit = b.m[3] == 0.0f && b.m[7] == 0.0f && b.m[11] == 0.0f && b.m[15] == 1.0f;
    if (unit) back_project_kernel<S, kMask, true><<<grid, block, 0, stream>>>(s, b, vol, mask, residual, ray_length);
    else back_project_kernel<S, kMask, false><<<grid, block, 0, stream>>>(s, b, vol, mask, residual, ray_length);
}

}  // namespace

void launch_forward_project(const SlabParams& s, const RayParams& r, etn_voxel_type vt, const void* volume,
                            const uint8_t* mask, float* projection, float* traversal_length, hipStream_t stream)
{
    if (!mask && plane_forward_project(s, r, vt, volume, projection, traversal_length, stream)) return;
#define ETN_FORWARD(S)                                                                                          \
    (mask ? forward_project_typed<S, true>(s, r, volume, mask, projection, traversal_length, stream)            \
          : forward_project_typed<S, false>(s, r, volume, mask, projection, traversal_length, stream))
    switch (vt) {
        case ETN_VOXEL_FLOAT32: ETN_FORWARD(F32); break;
        case ETN_VOXEL_FLOAT16: ETN_FORWARD(F16); break;
        case ETN_VOXEL_BFLOAT16: ETN_FORWARD(BF16); break;
    }
#undef ETN_FORWARD
    check_launch("forward projection launch");
}

void launch_back_project(const SlabParams& s, const BpParams& b, etn_voxel_type vt, void* volume,
                         const uint8_t* mask, const float* residual, const float* ray_length, hipStream_t stream)
{
    if (!mask && plane_back_project(s, b, vt, volume, residual, ray_length, stream)) return;
#define ETN_BACK(S)                                                                             \
    (mask ? back_project_typed<S, true>(s, b, volume, mask, residual, ray_length, stream)       \
          : back_project_typed<S, false>(s, b, volume, mask, residual, ray_length, stream))
    switch (vt) {
        case ETN_VOXEL_FLOAT32: ETN_BACK(F32); break;
        case ETN_VOXEL_FLOAT16: ETN_BACK(F16); break;
        case ETN_VOXEL_BFLOAT16: ETN_BACK(BF16); break;
    }
#undef ETN_BACK
    check_launch("back projection launch");
}

void launch_compare(uint32_t n, const void* real, etn_voxel_type real_type, const float* virt, float* residual,
                    hipStream_t stream)
{
    const uint32_t grid = (n + 255) / 256;
    if (real_type == ETN_VOXEL_FLOAT16)
        compare_kernel<F16><<<grid, 256, 0, stream>>>(n, (const __half*)real, virt, residual);
    else if (real_type == ETN_VOXEL_BFLOAT16)
        compare_kernel<BF16><<<grid, 256, 0, stream>>>(n, (const uint16_t*)real, virt, residual);
    else
        compare_kernel<F32><<<grid, 256, 0, stream>>>(n, (const float*)real, virt, residual);
    check_launch("compare launch");
}

void launch_compare(uint32_t n, const float* real, const float* virt, float* residual, hipStream_t stream)
{
    launch_compare(n, real, ETN_VOXEL_FLOAT32, virt, residual, stream);
}

void launch_long_object_compensate(uint32_t n, float* projection, float* length, float c, hipStream_t stream)
{
    loc_kernel<<<(n + 255) / 256, 256, 0, stream>>>(n, projection, length, c);
    check_launch("long object compensation launch");
}

void launch_ray_length(const float bmin[3], const float bmax[3], const RayParams& r, float* out, hipStream_t stream)
{
    const dim3 block(64, 4);
    const dim3 grid((r.nu + 63) / 64, (r.nv + 3) / 4);
    ray_length_kernel<<<grid, block, 0, stream>>>(r, bmin[0], bmin[1], bmin[2], bmax[0], bmax[1], bmax[2], out);
    check_launch("ray length launch");
}

void launch_ray_length_batch(const float bmin[3], const float bmax[3], const RayParams* params, uint32_t count,
                             uint32_t nu, uint32_t nv, float* out, size_t stride, hipStream_t stream)
{
    if (count == 0) return;
    if (count > 65535) fail("ray length: at most 65535 images per launch");
    const dim3 block(64, 4);
    const dim3 grid((nu + 63) / 64, (nv + 3) / 4, count);
    ray_length_batch_kernel<<<grid, block, 0, stream>>>(params, bmin[0], bmin[1], bmin[2], bmax[0], bmax[1], bmax[2],
                                                        out, stride);
    check_launch("ray length launch");
}

void launch_sum_squared_difference(const void* a, etn_voxel_type a_type, const float* b, size_t count,
                                   double* partials, double* out, hipStream_t stream)
{
    if (a_type == ETN_VOXEL_FLOAT16)
        ssd_partial_kernel<F16><<<kSsdBlocks, kSsdThreads, 0, stream>>>((const __half*)a, b, count, partials);
    else if (a_type == ETN_VOXEL_BFLOAT16)
        ssd_partial_kernel<BF16><<<kSsdBlocks, kSsdThreads, 0, stream>>>((const uint16_t*)a, b, count, partials);
    else
        ssd_partial_kernel<F32><<<kSsdBlocks, kSsdThreads, 0, stream>>>((const float*)a, b, count, partials);
    ssd_final_kernel<<<1, kSsdThreads, 0, stream>>>(partials, kSsdBlocks, out);
    check_launch("residual norm launch");
}

// Scratch of the allocation-free residual norm: the kSsdBlocks FP64 partial
// sums of ssd_partial_kernel (4 KiB), one copy per GPU, held by each GPU the
// library runs on until the process ends.  Host code never passes `scratch`
// itself to a kernel (on the host it names a stand-in, not device memory): it
// looks up each device's address once, with that device current, and uses it.
static __device__ __align__(256) double scratch[kSsdBlocks];

double* ssd_static_scratch(int device)
{
    static std::mutex lock;
    static std::vector<double*> address;   // per device, filled on first use
    std::lock_guard<std::mutex> guard(lock);
    if (device < 0) fail("residual norm scratch: invalid device");
    if ((size_t)device >= address.size()) address.resize((size_t)device + 1, nullptr);
    if (!address[device]) {
        int current = 0;
        ETN_HIP(hipGetDevice(&current));
        if (current != device) ETN_HIP(hipSetDevice(device));
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (current != device) ETN_HIP(hipSetDevice(current));
        ETN_HIP(e);
        if (!p) fail("residual norm scratch: no device address");
        address[device] = static_cast<double*>(p);
    }
    return address[device];
}

void launch_sum_squared_difference(const float* a, const float* b, size_t count, double* partials, double* out,
                                   hipStream_t stream)
{
    launch_sum_squared_difference(a, ETN_VOXEL_FLOAT32, b, count, partials, out, stream);
}

void launch_convert(const void* src, etn_voxel_type st, void* dst, etn_voxel_type dt, size_t count, hipStream_t stream)
{
    const uint32_t grid = grid_for(count, 256);
#define ETN_CONVERT(SS, DS)                                                                                    \
    convert_kernel<SS, DS><<<grid, 256, 0, stream>>>((const typename SS::T*)src, (typename DS::T*)dst, count)
    if (st == ETN_VOXEL_FLOAT32 && dt == ETN_VOXEL_FLOAT32) ETN_CONVERT(F32, F32);
    else if (st == ETN_VOXEL_FLOAT32 && dt == ETN_VOXEL_FLOAT16) ETN_CONVERT(F32, F16);
    else if (st == ETN_VOXEL_FLOAT32 && dt == ETN_VOXEL_BFLOAT16) ETN_CONVERT(F32, BF16);
    else if (st == ETN_VOXEL_FLOAT16 && dt == ETN_VOXEL_FLOAT32) ETN_CONVERT(F16, F32);
    else if (st == ETN_VOXEL_FLOAT16 && dt == ETN_VOXEL_FLOAT16) ETN_CONVERT(F16, F16);
    else if (st == ETN_VOXEL_FLOAT16 && dt == ETN_VOXEL_BFLOAT16) ETN_CONVERT(F16, BF16);
    else if (st == ETN_VOXEL_BFLOAT16 && dt == ETN_VOXEL_FLOAT32) ETN_CONVERT(BF16, F32);
    else if (st == ETN_VOXEL_BFLOAT16 && dt == ETN_VOXEL_FLOAT16) ETN_CONVERT(BF16, F16);
    else ETN_CONVERT(BF16, BF16);
#undef ETN_CONVERT
    check_launch("convert launch");
}

void launch_fill(void* dst, etn_voxel_type t, float value, size_t count, hipStream_t stream)
{
    const uint32_t grid = grid_for(count, 256);
    if (t == ETN_VOXEL_FLOAT32) fill_kernel<F32><<<grid, 256, 0, stream>>>((float*)dst, value, count);
    else if (t == ETN_VOXEL_FLOAT16) fill_kernel<F16><<<grid, 256, 0, stream>>>((__half*)dst, value, count);
    else fill_kernel<BF16><<<grid, 256, 0, stream>>>((uint16_t*)dst, value, count);
    check_launch("fill launch");
}

void launch_zero(float* dst, size_t count, hipStream_t stream)
{
    fill_kernel<F32><<<grid_for(count, 256), 256, 0, stream>>>(dst, 0.0f, count);
    check_launch("zero launch");
}

}  // namespace dev
}  // namespace etn
