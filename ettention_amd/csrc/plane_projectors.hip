// Single forward and back projections of single-axis tilt geometries, float
// operation for float operation those of the generic kernels (projectors.hip),
// so the results are bit-identical to theirs.
//
// When the rays and the detector's u axis have no y component and the v axis
// has nothing else, every ray of a detector row lies in one volume plane y = j,
// and the rays of one detector column take the same x-z steps in every plane.
// A workgroup then owns a few consecutive detector rows (their planes): the
// steps of a column are worked out once for all of them, and the voxels a
// thread reads are neighbours in LDS.  The back projection has the same
// structure: the detector column of a voxel depends on x and z only, its
// detector rows on y only.
#include <cfloat>
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "device_math.hpp"

namespace etn {
namespace dev {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// four consecutive voxels of one plane
template <typename S>
struct Quad;
template <>
struct Quad<F32> {
    using V = f32x4;
    static __device__ __forceinline__ void unpack(const V& v, float* o) { o[0] = v[0]; o[1] = v[1]; o[2] = v[2]; o[3] = v[3]; }
};
template <typename S16>
struct Quad16 {
    typedef uint32_t V __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ void unpack(const V& v, float* o)
    {
        S16::unpack2(v[0], o[0], o[1]);
        S16::unpack2(v[1], o[2], o[3]);
    }
};
template <>
struct Quad<F16> : Quad16<F16> {};
template <>
struct Quad<BF16> : Quad16<BF16> {};

// ---- forward projection ------------------------------------------------------
// P detector rows a workgroup.  The volume streams through LDS in bands of z
// rows, in the direction the rays travel in z, P planes interleaved voxel by
// voxel; the next band's loads are in flight while the rays cross this one.
// A thread traces kCols columns (512 apart), its state in registers across
// bands: 12 VALU instructions a step for all P planes (which the generic kernel
// spends, and a dependent gather from memory, on each ray).
// Bound by the volume's read: 512^3 f32 in 0.10 ms (5.1 TB/s, the rate of a
// large copy), 1.39 ms on the generic kernel.
constexpr int kFpThreads = 512;
constexpr int kFpLds = 16384;       // floats: two workgroups of 64 KiB a CU

// State of a detector column: distances to the next x and z border, position as
// a byte offset in the interleaved planes, x steps left inside the volume.
template <int P>
struct ColumnRay {
    float rx, rz, stepx, stepz;
    int at, left, dx, dz;
    float acc[P], len;
};

template <int P>
struct Lanes;
template <>
struct Lanes<1> {
    using V = float;
    static __device__ __forceinline__ float get(const V& v, int) { return v; }
};
template <>
struct Lanes<2> {
    using V = float2;
    static __device__ __forceinline__ float get(const V& v, int p) { return p ? v.y : v.x; }
};

template <>
struct Lanes<4> {
    using V = f32x4;
    static __device__ __forceinline__ float get(const V& v, int p) { return v[p]; }
};

// P planes' four voxels each, interleaved, as 16-byte LDS cells
template <int P>
__device__ __forceinline__ void interleave(const float (*v)[4], f32x4* to)
{
    if constexpr (P == 1) {
        to[0] = f32x4{v[0][0], v[0][1], v[0][2], v[0][3]};
    } else if constexpr (P == 2) {
        to[0] = f32x4{v[0][0], v[1][0], v[0][1], v[1][1]};
        to[1] = f32x4{v[0][2], v[1][2], v[0][3], v[1][3]};
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) to[i] = f32x4{v[0][i], v[1][i], v[2][i], v[3][i]};
    }
}

template <typename S, bool kVec, int P, int kCols>
__global__ void __launch_bounds__(kFpThreads, kCols == 1 ? 4 : 2)
    plane_forward_kernel(SlabParams s, RayParams g, const typename S::T* vol, float* proj, float* len, int band)
{
    using Q = Quad<S>;
    using L = Lanes<P>;
    __shared__ __attribute__((aligned(16))) float lds[kFpLds];
    const int tid = threadIdx.x;
    const int row0 = blockIdx.x * P, rows = min(P, (int)g.nv - row0);
    const int nx = s.res[0], nz = s.res[2], nu = (int)g.nu;
    const DdaConst c = dda_const(g.ray, s.vs);
    // the y part of dda_begin for each row: its plane, or none
    int plane[P];
    bool hit[P];
    bool any = false;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        float src[3];
        fp_ray_source(g, 0, (uint32_t)min(row0 + p, (int)g.nv - 1), 0, 0, 1.0f, 0.5f, src);
        const float t0 = (s.bmin[1] - src[1]) * c.inv[1], t1 = (s.bmax[1] - src[1]) * c.inv[1];
        hit[p] = p < rows && fminf(t0, t1) < 0.0f && fmaxf(t0, t1) > 0.0f;
        const float y = fminf(fmaxf(src[1], s.bmin[1]), s.bmax[1]);
        plane[p] = min(max((int)((y - s.bmin[1]) * (1.0f / s.vs[1])), 0), s.res[1] - 1);
        any = any || hit[p];
    }

    ColumnRay<P> ray[kCols];
#pragma unroll
    for (int k = 0; k < kCols; ++k) {
        const int u = k * kFpThreads + tid;
        ColumnRay<P>& r = ray[k];
        r.left = 0;
        r.at = 0;
        r.len = 0.0f;
#pragma unroll
        for (int p = 0; p < P; ++p) r.acc[p] = 0.0f;
        if (any && u < nu) {
            // dda_begin in x and z; a ray whose row is inside the volume in y
            // has y entry and exit beyond every other (checked on the host)
            float src[3];
            fp_ray_source(g, (uint32_t)u, (uint32_t)row0, 0, 0, 1.0f, 0.5f, src);
            SlabParams flat = s;
            src[1] = 0.0f;
            flat.bmin[1] = -1.0f;
            flat.bmax[1] = 1.0f;
            DdaRay d;
            dda_begin(flat, c, src, d);
            r.rx = d.res[0];
            r.rz = d.res[2];
            r.stepx = c.step[0];
            r.stepz = c.step[2];
            r.at = (d.vox[2] * nx + d.vox[0]) * P * 4;
            r.left = !d.live ? 0 : c.sign[0] > 0 ? nx - d.vox[0] : c.sign[0] < 0 ? d.vox[0] + 1 : 0x7fffffff;
            r.dx = c.sign[0] * P * 4;
            r.dz = c.sign[2] * nx * P * 4;
        }
    }

    if (any) {
        const size_t slice = (size_t)s.nx * s.ny;
        const typename S::T* base[P];
#pragma unroll
        for (int p = 0; p < P; ++p) base[p] = vol + s.first_voxel + (size_t)plane[p] * s.nx;
        const int bands = (nz + band - 1) / band, quads = nx / 4;
        constexpr int kItems = kVec ? kFpLds / (4 * P * kFpThreads) : 1;
        typename Q::V pre[kItems][P];
        auto range = [&](int b, int& z0, int& z1) {
            z0 = (c.sign[2] >= 0 ? b : bands - 1 - b) * band;
            z1 = min(z0 + band, nz);
        };
        auto load = [&](int z0, int z1) {
            if constexpr (kVec) {
                const int n = (z1 - z0) * quads;
#pragma unroll
                for (int k = 0; k < kItems; ++k) {
                    const int i = min(k * kFpThreads + tid, n - 1), z = i / quads, x = (i - z * quads) * 4;
#pragma unroll
                    for (int p = 0; p < P; ++p)
                        pre[k][p] = __builtin_nontemporal_load(
                            reinterpret_cast<const typename Q::V*>(base[p] + (size_t)(z0 + z) * slice + x));
                }
            }
        };
        int z0, z1;
        range(0, z0, z1);
        load(z0, z1);
        for (int b = 0; b < bands; ++b) {
            range(b, z0, z1);
            if constexpr (kVec) {
                const int n = (z1 - z0) * quads;
#pragma unroll
                for (int k = 0; k < kItems; ++k) {
                    const int i = k * kFpThreads + tid;
                    if (i < n) {
                        float v[P][4];
#pragma unroll
                        for (int p = 0; p < P; ++p) Q::unpack(pre[k][p], v[p]);
                        interleave<P>(v, reinterpret_cast<f32x4*>(lds) + (size_t)i * P);
                    }
                }
            } else {
                const int n = (z1 - z0) * nx;
#pragma unroll 4
                for (int i = tid; i < n; i += kFpThreads) {
                    const int z = i / nx, x = i - z * nx;
#pragma unroll
                    for (int p = 0; p < P; ++p) lds[i * P + p] = S::load(base[p], (size_t)(z0 + z) * slice + x);
                }
            }
            int n0 = 0, n1 = 0;
            if (b + 1 < bands) {
                range(b + 1, n0, n1);
                load(n0, n1);
            }
            __syncthreads();
            const unsigned bytes = (unsigned)((z1 - z0) * nx * P) * 4u;
            const int start = z0 * nx * P * 4;
            const char* rows_at = reinterpret_cast<const char*>(lds);
#pragma unroll
            for (int k = 0; k < kCols; ++k) {
                ColumnRay<P>& r = ray[k];
                int at = r.at - start, left = r.left;
                float rx = r.rx, rz = r.rz;
                // the voxel of a step is read one step ahead: its address does
                // not depend on any voxel (past the band's end: its last voxel)
                const unsigned end = bytes - 4u * P;
                typename L::V next = *reinterpret_cast<const typename L::V*>(rows_at + min((unsigned)at, end));
                while (left != 0 && (unsigned)at < bytes) {
                    const typename L::V v = next;
                    const bool ix = rx <= rz;
                    const float dt = ix ? rx : rz, rest = fabsf(rx - rz);   // the axis not stepped loses dt
                    rx = ix ? r.stepx : rest;
                    rz = ix ? rest : r.stepz;
                    at += ix ? r.dx : r.dz;
                    left -= ix ? 1 : 0;
                    next = *reinterpret_cast<const typename L::V*>(rows_at + min((unsigned)at, end));
#pragma unroll
                    for (int p = 0; p < P; ++p) r.acc[p] += dt * L::get(v, p);
                    r.len += dt;
                }
                r.at = at + start;
                r.left = left;
                r.rx = rx;
                r.rz = rz;
            }
            __syncthreads();
        }
    }

#pragma unroll
    for (int k = 0; k < kCols; ++k) {
        const int u = k * kFpThreads + tid;
        if (u >= nu) continue;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            if (p >= rows) continue;
            const size_t i = (size_t)(row0 + p) * nu + u;
            const float acc = 0.0f + (hit[p] ? ray[k].acc[p] : 0.0f), l = 0.0f + (hit[p] ? ray[k].len : 0.0f);
            proj[i] += acc / 1.0f;
            len[i] += l / 1.0f;
        }
    }
}

template <typename S, bool kVec, int P>
void launch_forward_cols(const SlabParams& s, const RayParams& r, const void* vol, float* proj, float* len, int band,
                         hipStream_t stream)
{
    const dim3 grid((r.nv + P - 1) / P);
    const auto* v = static_cast<const typename S::T*>(vol);
    if (r.nu <= (uint32_t)kFpThreads)
        plane_forward_kernel<S, kVec, P, 1><<<grid, kFpThreads, 0, stream>>>(s, r, v, proj, len, band);
    else if (r.nu <= 2u * kFpThreads)
        plane_forward_kernel<S, kVec, P, 2><<<grid, kFpThreads, 0, stream>>>(s, r, v, proj, len, band);
    else
        plane_forward_kernel<S, kVec, P, 4><<<grid, kFpThreads, 0, stream>>>(s, r, v, proj, len, band);
}

// rows read four voxels at a time
bool vector_rows(const SlabParams& s, const void* vol, size_t voxel)
{
    return s.res[0] % 4 == 0 && s.nx % 4 == 0 && reinterpret_cast<uintptr_t>(vol) % (4 * voxel) == 0;
}

template <typename S>
void launch_forward_typed(const SlabParams& s, const RayParams& r, const void* vol, float* proj, float* len,
                          hipStream_t stream)
{
    const int nx = s.res[0];
    const bool vec = vector_rows(s, vol, sizeof(typename S::T));
    // two rows a workgroup halve the steps' instructions; one row gives twice
    // the workgroups, where two would not reach every CU (256 of them)
    const bool two = r.nv >= 512 && nx * 2 <= kFpLds;
    const int band = std::max(1, std::min(s.res[2], kFpLds / (nx * (two ? 2 : 1))));
    if (two && vec) launch_forward_cols<S, true, 2>(s, r, vol, proj, len, band, stream);
    else if (two) launch_forward_cols<S, false, 2>(s, r, vol, proj, len, band, stream);
    else if (vec) launch_forward_cols<S, true, 1>(s, r, vol, proj, len, band, stream);
    else launch_forward_cols<S, false, 1>(s, r, vol, proj, len, band, stream);
}

// Whether a geometry's rows lie in planes and take the same steps in each.
// (sub: the rows are sub-ray rows, so many a pixel)
bool plane_geometry_fits(const SlabParams& s, const RayParams& r, int sub = 1)
{
    if (r.nu == 0 || r.nv == 0 || s.res[0] > kFpLds) return false;
    if (r.ray[1] != 0.0f || r.h[1] != 0.0f || r.v[0] != 0.0f || r.v[2] != 0.0f) return false;
    // the 2048-step limit cannot bind, and no ray's y interval decides where
    // it enters or leaves: a row's interval runs beyond +-1e30 (inside the
    // volume) or lies wholly beyond (outside), x and z times stay far below
    if (s.res[0] + s.res[2] > 2040) return false;
    if ((size_t)s.res[0] * s.res[2] > (size_t)1 << 27) return false;
    float size = 0.0f;
    for (int k = 0; k < 3; k += 2) {
        const float big = std::fmax(std::fabs(s.bmin[k]), std::fabs(s.bmax[k])) + std::fabs(r.source[k]) +
                          std::fabs(r.h[k]) * (float)r.nu;
        if (!(big < 1e8f)) return false;
        size = std::fmax(size, std::fabs(r.ray[k]));
    }
    if (!(size > 0.5f)) return false;   // (a unit vector without y) the larger of x and z bounds the times
    const float inv = -FLT_MAX;
    const float sd = 1.0f / (float)sub, off = sd / 2.0f;
    const uint32_t rows = r.nv * (uint32_t)sub;
    auto source_y = [&](uint32_t y) {
        const float fy = (float)(y / sub) + off + sd * (float)(y % sub);
        const float rv = r.v[1] * fy;
        return r.source[1] + 0.0f + rv;
    };
    if (!std::isfinite(source_y(0)) || !std::isfinite(source_y(rows - 1))) return false;
    // a row's source moves one way with the row (each operation rounds
    // monotonically), so if any row lies too near a face of the box, the first, the
    // last or one beside the face does
    for (const float face : {s.bmin[1], s.bmax[1]}) {
        const bool above = face - source_y(0) > 0.0f;
        uint32_t lo = 0, hi = rows;     // first row on the other side of the face than row 0
        while (lo < hi) {
            const uint32_t mid = (lo + hi) / 2;
            if ((face - source_y(mid) > 0.0f) == above) lo = mid + 1;
            else hi = mid;
        }
        for (const uint32_t y : {0u, lo > 0 ? lo - 1 : 0u, std::min(lo, rows - 1), rows - 1}) {
            const float t = (face - source_y(y)) * inv;
            if (!(std::fabs(t) > 1e30f)) return false;
        }
    }
    return true;
}

// Whether plane_forward_kernel computes what forward_project_kernel does.
bool plane_forward_fits(const SlabParams& s, const RayParams& r)
{
    return r.samples == 1 && r.nu <= 4u * kFpThreads && plane_geometry_fits(s, r);
}

// ---- back projection ----------------------------------------------------------
// P planes x 256 columns (128 or 64 where those fit nx better, with 2 or 4 rows of
// threads for slices in turn) x `depth` slices a workgroup, one voxel a thread and
// step.  The plane's two detector rows over the columns the
// workgroup's voxels project to are staged in LDS as (value, difference) pairs,
// residual and length apart, zero beyond the detector; neighbouring lanes then
// read neighbouring 16-byte records.  Column and weight of a voxel are worked
// out once for the P planes.  Bound by the volume's read and write: 512^3 f32
// in 0.21 ms (5.1 TB/s), 0.77 ms on the generic kernel.
constexpr int kBpThreads = 256;
constexpr int kBpPlanes = 4;
constexpr int kBpColumns = 312;     // staged columns: 39 KiB, four workgroups a CU
constexpr int kBpUnroll = 4;        // slices in flight

template <typename S>
__global__ void __launch_bounds__(kBpThreads, 4)
    plane_back_kernel(SlabParams s, BpParams b, typename S::T* vol, const float* residual, const float* length, int depth,
                      int shift)
{
    __shared__ f32x4 rec[kBpPlanes][2][kBpColumns];   // {r0, dr0, r1, dr1}, {l0, dl0, l1, dl1} of a column
    __shared__ float weight[kBpPlanes];               // ty of each plane
    const int tid = threadIdx.x, wide = 1 << shift;   // columns, a wave or more
    const int x0 = blockIdx.x * wide, y0 = blockIdx.y * kBpPlanes, z0 = blockIdx.z * depth;
    const int x1 = min(x0 + wide, s.res[0]), z1 = min(z0 + depth, s.res[2]);
    const int planes = min(kBpPlanes, s.res[1] - y0);
    const float m0 = b.m[0], m4 = b.m[4], m8 = b.m[8], m12 = b.m[12];
    const float4 smp = b.samples[0];
    const int nu = (int)b.nu, nv = (int)b.nv;
    // detector columns the workgroup's voxels reach (u is linear in x and z),
    // one more on each side for its rounding
    auto column = [&](int x, int z) {
        const float px = s.bmin[0] + ((float)x + 0.5f) * s.vs[0] + smp.x, pz = s.bmin[2] + ((float)z + 0.5f) * s.vs[2] + smp.z;
        return m0 * px + m8 * pz + m12 - 0.5f;
    };
    const float ua = column(x0, z0), ub = column(x1 - 1, z0), uc = column(x0, z1 - 1), ud = column(x1 - 1, z1 - 1);
    const float umin = fminf(fminf(ua, ub), fminf(uc, ud)), umax = fmaxf(fmaxf(ua, ub), fmaxf(uc, ud));
    // (clamped: columns left of -2 and right of nu read zeros like those)
    const int first = min((int)floorf(fminf(fmaxf(umin, -2.0f), (float)nu + 2.0f)) - 1, nu);
    const int count = max(min((int)floorf(fmaxf(fminf(umax, (float)nu), -2.0f)) + 2 - first, kBpColumns), 1);
    for (int e = tid; e < kBpPlanes * kBpColumns; e += kBpThreads) {
        const int p = e / kBpColumns, k = e - p * kBpColumns, u = first + k;
        if (p >= planes || k >= count) continue;
        const float py = s.bmin[1] + ((float)(y0 + p) + 0.5f) * s.vs[1] + smp.y;
        float v = b.m[1] * 0.0f + b.m[5] * py;
        v = v + b.m[9] * 0.0f;
        v = v + b.m[13] * 1.0f;
        float base;
        const float ty = cl_fract(v - 0.5f, &base);
        const int row = (int)base;
        float o[2][4];
        for (int r = 0; r < 2; ++r) {
            const bool rok = row + r >= 0 && row + r < nv;
            const bool ok0 = rok && u >= 0 && u < nu, ok1 = rok && u + 1 >= 0 && u + 1 < nu;
            const size_t at = (size_t)(row + r) * nu + u;
            const float r0 = ok0 ? residual[at] : 0.0f, r1 = ok1 ? residual[at + 1] : 0.0f;
            const float l0 = ok0 ? length[at] : 0.0f, l1 = ok1 ? length[at + 1] : 0.0f;
            o[0][2 * r] = r0;
            o[0][2 * r + 1] = r1 - r0;
            o[1][2 * r] = l0;
            o[1][2 * r + 1] = l1 - l0;
        }
        rec[p][0][k] = f32x4{o[0][0], o[0][1], o[0][2], o[0][3]};
        rec[p][1][k] = f32x4{o[1][0], o[1][1], o[1][2], o[1][3]};
        if (k == 0) weight[p] = ty;
    }
    __syncthreads();
    const int x = x0 + (tid & (wide - 1));
    if (x >= x1) return;
    float ty[kBpPlanes];
#pragma unroll
    for (int p = 0; p < kBpPlanes; ++p) ty[p] = p < planes ? weight[p] : 0.0f;
    const float px = (s.bmin[0] + ((float)x + 0.5f) * s.vs[0]) + smp.x;
    const float xt = m0 * px + m4 * 0.0f;   // m4 = 0: the y term adds a zero
    const size_t slice = (size_t)s.nx * s.ny;
    typename S::T* at = vol + s.first_voxel + (size_t)y0 * s.nx + x;
    const int first_z = z0 + __builtin_amdgcn_readfirstlane(tid >> shift) * kBpUnroll;
    for (int z = first_z; z < z1; z += kBpUnroll * (kBpThreads >> shift)) {
        float value[kBpUnroll][kBpPlanes];
#pragma unroll
        for (int j = 0; j < kBpUnroll; ++j)
#pragma unroll
            for (int p = 0; p < kBpPlanes; ++p)
                if (z + j < z1 && p < planes) value[j][p] = S::load(at, (size_t)(z + j) * slice + (size_t)p * s.nx);
#pragma unroll
        for (int j = 0; j < kBpUnroll; ++j) {
            if (z + j >= z1) break;
            const float pz = (s.bmin[2] + ((float)(z + j) + 0.5f) * s.vs[2]) + smp.z;
            float u = xt + m8 * pz;
            u = u + m12 * 1.0f;
            float base;
            const float tx = cl_fract(u - 0.5f, &base);
            const int k = min(max((int)base - first, 0), count - 1);
#pragma unroll
            for (int p = 0; p < kBpPlanes; ++p) {
                if (p >= planes) break;
                const f32x4 ll = rec[p][1][k], rr = rec[p][0][k];
                const float L0 = ll[0] + ll[1] * tx, L1 = ll[2] + ll[3] * tx, L = L0 + (L1 - L0) * ty[p];
                const float R0 = rr[0] + rr[1] * tx, R1 = rr[2] + rr[3] * tx, R = R0 + (R1 - R0) * ty[p];
                if (L > kEpsilon) value[j][p] += 0.0f + R * b.lambda * (smp.w / L);
                S::store(at, (size_t)(z + j) * slice + (size_t)p * s.nx, value[j][p]);
            }
        }
    }
}

// u of x and z alone, v of y alone, no perspective, coordinates well inside
// float's whole numbers.
bool single_axis_matrix(const SlabParams& s, const BpParams& b)
{
    const float* m = b.m;
    if (b.nu == 0 || b.nv == 0) return false;
    if (m[4] != 0.0f || m[1] != 0.0f || m[9] != 0.0f) return false;
    if (m[3] != 0.0f || m[7] != 0.0f || m[11] != 0.0f || m[15] != 1.0f) return false;
    for (int k = 0; k < 16; ++k)
        if (!std::isfinite(m[k])) return false;
    for (int k = 0; k < 3; ++k)
        if (!(std::fabs(s.bmin[k]) < 1e5f && std::fabs(s.bmax[k]) < 1e5f)) return false;
    return std::fabs(m[0]) + std::fabs(m[8]) < 8.0f && std::fabs(m[12]) < 1e5f && std::fabs(m[5]) < 8.0f &&
           std::fabs(m[13]) < 1e5f;
}

// Columns (their log2) and slices of a workgroup of plane_back_kernel; depth 0
// where it does not compute what back_project_kernel does.
struct BackTile {
    int shift = 8, depth = 0;
};
BackTile plane_back_tile(const SlabParams& s, const BpParams& b)
{
    BackTile t;
    const float* m = b.m;
    if (b.nsamples != 1 || !single_axis_matrix(s, b)) return t;
    // the widest rows of those that leave the fewest columns idle (260^3 bf16 at 60
    // degrees: 0.110 ms with rows of 256, 0.100 on the generic kernel, 0.066 with 64)
    auto padded = [&](int shift) { return (s.res[0] + (1 << shift) - 1) >> shift << shift; };
    for (int shift = 7; shift >= 6; --shift)
        if (padded(shift) < padded(t.shift)) t.shift = shift;
    const int wide = 1 << t.shift;
    const int tiles = (padded(t.shift) >> t.shift) * ((s.res[1] + kBpPlanes - 1) / kBpPlanes);
    if ((s.res[1] + kBpPlanes - 1) / kBpPlanes > 65535) return t;
    // as deep as the columns fit, at most 64 slices, less where that leaves
    // fewer workgroups than the CUs hold (four each), but some for every wave
    const int least = std::max(8, kBpUnroll * (kBpThreads >> t.shift));
    int depth = 64;
    while (depth > least && tiles * ((s.res[2] + depth - 1) / depth) < 1024) depth /= 2;
    for (; depth >= 4; depth /= 2) {
        const float columns = std::fabs(m[0]) * s.vs[0] * (float)std::min(wide, s.res[0]) +
                              std::fabs(m[8]) * s.vs[2] * (float)depth + 6.0f;
        if (columns <= (float)kBpColumns && (s.res[2] + depth - 1) / depth <= 65535) {
            t.depth = depth;
            return t;
        }
    }
    return t;
}

// ---- back projection of many projections in one sweep ---------------------------
// The arithmetic of the fused kernels' back projection (bp_update_fast): A + B tx
// from columns whose row pair is interpolated at staging, the hardware
// reciprocal of the ray length.  A workgroup owns kSweepPlanes planes x 64
// columns x 64 slices, held in registers (16 slices a wave) while every
// projection is applied in turn, so that the volume is read and written once
// for all of them.  Column, weight and LDS address of a voxel are the same in
// every plane: 8 of the 13.5 VALU instructions of an update.  kEqual: the
// detector rows of the workgroup's planes have equal ray lengths too (rows of
// rays that all cross the volume; the host knows them), then the reciprocal is
// shared and 3 instructions per update and plane remain.
// A projection's columns (the 64 x 64 tile reaches at most 97 at unit pitch) are
// loaded while the one before it is applied and staged in alternating buffers.
// Bound by VALU issue (busy 0.67 of the time by its counter) and the record reads
// together: 0.071 ms a projection at 512^3 on the fused kernels (eight a sweep),
// 0.037 to 0.039 here.
constexpr int kSweepThreads = 256;
constexpr int kSweepPlanes = 4;
constexpr int kSweepDepth = 16;      // slices a wave
constexpr int kSweepTile = 64;       // columns, and slices of the four waves
constexpr int kSweepColumns = 128;   // staged detector columns: one a pair of threads

// the planes' values rounded to storage, two in a conversion
template <typename S>
__device__ __forceinline__ void round_planes(float* v)
{
    if constexpr (sizeof(typename S::T) == 2) {
#pragma unroll
        for (int p = 0; p < kSweepPlanes; p += 2) {
            const uint32_t packed = S::pack2(v[p], v[p + 1]);
            S::unpack2(packed, v[p], v[p + 1]);
        }
    }
}

struct SweepLds {
    f32x4 ab[2][2][kSweepColumns];    // {A, B} of planes 0 and 1, of planes 2 and 3
    f32x4 ll[2][2][kSweepColumns];    // the same of the ray lengths
    float2 lu[2][kSweepColumns];      // of every plane's ray lengths (kEqual)
    f32x4 zterm[2][kSweepTile / 4];
};

template <typename S, bool kEqual>
__device__ __forceinline__ void sweep_back(SweepLds& lds, const SlabParams& s, const BackView* __restrict__ views, int n,
                                           typename S::T* vol, int nu, int nv, int group)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int x0 = blockIdx.x * kSweepTile, y0 = group * kSweepPlanes, z0 = blockIdx.z * kSweepTile;
    const int x = x0 + lane, zw = z0 + wave * kSweepDepth;
    const int planes = min(kSweepPlanes, s.res[1] - y0);
    const bool xin = x < s.res[0];
    const size_t slice = (size_t)s.nx * s.ny;
    typename S::T* base = vol + s.first_voxel + (size_t)zw * slice + (size_t)y0 * s.nx;

    float value[kSweepDepth][kSweepPlanes];
#pragma unroll
    for (int j = 0; j < kSweepDepth; ++j)
#pragma unroll
        for (int p = 0; p < kSweepPlanes; ++p) {
            value[j][p] = 0.0f;
            if (zw + j < s.res[2] && p < planes && xin)
                value[j][p] = S::load(base + (size_t)j * slice + (size_t)p * s.nx, (size_t)(uint32_t)x);
        }
    const float xc = s.bmin[0] + ((float)x + 0.5f) * s.vs[0];

    // staging: thread 2 k + h takes column k of planes 2 h and 2 h + 1, whose
    // detector rows are the same for every projection (the host checks it)
    const int k = tid >> 1, h = tid & 1;
    uint32_t row0[2], row1[2];   // the planes' rows as byte offsets (clamped into the image)
    float ty[2];
    bool rin[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const BackView& v = views[0];
        const float py = s.bmin[1] + ((float)(y0 + 2 * h + i) + 0.5f) * s.vs[1];
        float vp = v.m5 * (py + v.sy);
        vp = vp + v.m13 * 1.0f;
        float base_row;
        ty[i] = cl_fract(vp - 0.5f, &base_row);
        const int row = (int)base_row;
        rin[i][0] = row >= 0 && row < nv;
        rin[i][1] = row + 1 >= 0 && row + 1 < nv;
        row0[i] = 4u * (uint32_t)(min(max(row, 0), nv - 1) * nu);
        row1[i] = 4u * (uint32_t)(min(max(row + 1, 0), nv - 1) * nu);
    }
    // the tile's corners
    const float cxa = s.bmin[0] + ((float)x0 + 0.5f) * s.vs[0], cxb = s.bmin[0] + ((float)(x0 + kSweepTile - 1) + 0.5f) * s.vs[0];
    const float cza = s.bmin[2] + ((float)z0 + 0.5f) * s.vs[2], czb = s.bmin[2] + ((float)(z0 + kSweepTile - 1) + 0.5f) * s.vs[2];
    const float zc = s.bmin[2] + ((float)(z0 + (tid & (kSweepTile - 1))) + 0.5f) * s.vs[2];

    float in[2][8];      // per plane: residual row, row + 1 at u and u + 1, the same of the lengths
    int first = 0;       // detector column 0 of the projection in the registers
    // (addresses are clamped into the images; what lies outside them is zeroed
    // at commit, so that nothing waits for a load before it is needed)
    auto load = [&](int q) {
        const BackView& v = views[q];
        const float m0 = v.m0, m8 = v.m8;
        // the tile's smallest u, less one for its rounding
        const float umin = m0 * ((m0 >= 0.0f ? cxa : cxb) + v.sx) + m8 * ((m8 >= 0.0f ? cza : czb) + v.sz) + v.m12 - 0.5f;
        first = (int)floorf(umin) - 1;
        const int u = first + k;
        const uint32_t k0 = 4u * (uint32_t)min(max(u, 0), nu - 1), k1 = 4u * (uint32_t)min(max(u + 1, 0), nu - 1);
        const char* res = reinterpret_cast<const char*>(v.residual);
        const char* len = reinterpret_cast<const char*>(v.length);
        auto at = [](const char* image, uint32_t offset) { return *reinterpret_cast<const float*>(image + offset); };
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            in[i][0] = at(res, row0[i] + k0);
            in[i][1] = at(res, row0[i] + k1);
            in[i][2] = at(res, row1[i] + k0);
            in[i][3] = at(res, row1[i] + k1);
            if (kEqual && i == 1) continue;   // (only plane 0's are kept)
            in[i][4] = at(len, row0[i] + k0);
            in[i][5] = at(len, row0[i] + k1);
            if (kEqual) continue;             // equal rows interpolate to themselves whatever the weight
            in[i][6] = at(len, row1[i] + k0);
            in[i][7] = at(len, row1[i] + k1);
        }
    };
    auto commit = [&](int q, int buf) {
        const BackView& v = views[q];
        const float weight = v.weight;
        const int u = first + k;
        const bool c0 = (unsigned)u < (unsigned)nu, c1 = (unsigned)(u + 1) < (unsigned)nu;
        f32x4 r, l;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            float e[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                if (t >= 4 && kEqual && (i == 1 || t >= 6)) continue;
                const bool row_in = kEqual || rin[i][t >> 1 & 1];   // (rows of one class lie on the detector)
                e[t] = row_in && (t & 1 ? c1 : c0) ? in[i][t] : 0.0f;
            }
            const float dr0 = e[1] - e[0], dr1 = e[3] - e[2];
            r[2 * i] = weight * fmaf(e[2] - e[0], ty[i], e[0]);
            r[2 * i + 1] = weight * fmaf(dr1 - dr0, ty[i], dr0);
            if constexpr (kEqual) {
                if (i == 0 && h == 0) lds.lu[buf][k] = make_float2(e[4], e[5] - e[4]);
            } else {
                const float dl0 = e[5] - e[4], dl1 = e[7] - e[6];
                l[2 * i] = fmaf(e[6] - e[4], ty[i], e[4]);
                l[2 * i + 1] = fmaf(dl1 - dl0, ty[i], dl0);
            }
        }
        lds.ab[buf][h][k] = r;
        if constexpr (!kEqual) lds.ll[buf][h][k] = l;
        if (tid < kSweepTile) reinterpret_cast<float*>(lds.zterm[buf])[tid] = v.m8 * (zc + v.sz);
    };
    load(0);
    commit(0, 0);
    for (int q = 0; q < n; ++q) {
        const int buf = q & 1, from = first;
        const BackView& v = views[q];
        const float xt = v.m0 * (xc + v.sx) + 0.0f, m12 = v.m12;
        __syncthreads();
        if (q + 1 < n) load(q + 1);
        const f32x4* rec = lds.ab[buf][0] - from;
        // u = ((m0 px + m4 py) + m8 pz) + m12, m4 = 0 (bp_update_fast)
        auto column = [&](float zt, float& tx) {
            float u = xt + zt;
            u = u + m12 * 1.0f;
            u = u - 0.5f;
            tx = __builtin_amdgcn_fractf(u);
            int i;
            asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(i) : "v"(u));
            return i;
        };
#pragma unroll
        for (int j = 0; j < kSweepDepth; ++j) {
            float tx;
            const int i = column(lds.zterm[buf][wave * (kSweepDepth / 4) + j / 4][j % 4], tx);
            const f32x4 a = rec[i], b = rec[i + kSweepColumns];
            const float r[kSweepPlanes] = {fmaf(a[1], tx, a[0]), fmaf(a[3], tx, a[2]), fmaf(b[1], tx, b[0]),
                                           fmaf(b[3], tx, b[2])};
            if constexpr (kEqual) {
                const float2 c = (lds.lu[buf] - from)[i];
                const float L = fmaf(c.y, tx, c.x);
                if (L > kEpsilon) {
                    const float inv = __builtin_amdgcn_rcpf(L);
#pragma unroll
                    for (int p = 0; p < kSweepPlanes; ++p) value[j][p] += r[p] * inv;
                }
            } else {
                const f32x4* len = lds.ll[buf][0] - from;
                const f32x4 c = len[i], d = len[i + kSweepColumns];
                const float L[kSweepPlanes] = {fmaf(c[1], tx, c[0]), fmaf(c[3], tx, c[2]), fmaf(d[1], tx, d[0]),
                                               fmaf(d[3], tx, d[2])};
                // (the branch also keeps the next slices' reads behind this one's updates)
                if (fmaxf(fmaxf(L[0], L[1]), fmaxf(L[2], L[3])) > kEpsilon) {
#pragma unroll
                    for (int p = 0; p < kSweepPlanes; ++p) {
                        const float next = value[j][p] + r[p] * __builtin_amdgcn_rcpf(L[p]);
                        value[j][p] = L[p] > kEpsilon ? next : value[j][p];
                    }
                }
            }
            round_planes<S>(value[j]);
            // one slice's reads in flight: all of them would take 10 VGPRs each
            __builtin_amdgcn_sched_barrier(0);
        }
        if (q + 1 < n) commit(q + 1, buf ^ 1);
    }
#pragma unroll
    for (int j = 0; j < kSweepDepth; ++j)
#pragma unroll
        for (int p = 0; p < kSweepPlanes; ++p)
            if (zw + j < s.res[2] && p < planes && xin)
                S::store(base + (size_t)j * slice + (size_t)p * s.nx, (size_t)(uint32_t)x, value[j][p]);
}

// The groups outside [equal0, equal1) first: they take longer.
template <typename S>
__global__ void __launch_bounds__(kSweepThreads, 3)
    sweep_back_kernel(SlabParams s, const BackView* __restrict__ views, int n, typename S::T* vol, int nu, int nv,
                      int equal0, int equal1)
{
    __shared__ SweepLds lds;
    const int others = (int)gridDim.y - (equal1 - equal0), i = blockIdx.y;
    if (i >= others) sweep_back<S, true>(lds, s, views, n, vol, nu, nv, equal0 + i - others);
    else sweep_back<S, false>(lds, s, views, n, vol, nu, nv, i < equal0 ? i : i + (equal1 - equal0));
}

// ---- forward projections of several projections in one sweep -----------------------
// plane_forward_kernel for up to kSweepForward projections of one z direction, P
// rows a workgroup, with fused multiply-adds (the fused kernels' fast arithmetic)
// and the residual written.  A thread traces up to eight ray columns, (projection,
// column, sub-ray column) triples, each through the P planes at once: 11
// instructions a step for the path and 1 for each plane's sum, where a ray a
// plane takes 12.  kMask: the ray length sums the voxels' mask weights, staged
// behind the P values of a voxel.  The columns are spread over several
// workgroups (slices), which read the same planes on the same XCD.  512 x 512 x
// 256, eight projections: 0.17 ms, VALU busy 0.54 of it, LDS bank conflicts 0.36;
// 250 x 300 x 150 bf16 with a mask and 4 x 4 sub-rays: 0.042 ms (0.055 with an index
// division for every staged voxel; reads of four steps in flight gained nothing).
template <bool kMask, int P>
struct SweepRay {
    float rx, rz, stepx, stepz;
    int at, left, dx, dz;
    float acc[P], len[kMask ? P : 1];
};

struct SweepForward {
    const ForwardView* views;
    int n, zdir, nu, nv;
    int sub, shift;      // sub-rays a pixel axis, log2 of the ray columns a pixel
    const uint8_t* mask;
    int band, groups;
};

template <typename S, bool kVec, bool kMask, int P, int R>
__global__ void __launch_bounds__(kFpThreads, R <= 4 ? 4 : 2)
    sweep_forward_kernel(SlabParams s, SweepForward a, const typename S::T* vol)
{
    using Q = Quad<S>;
    constexpr int W = kMask ? 2 * P : P;     // floats a voxel
    using L = Lanes<W>;
    constexpr int T = kFpThreads;
    __shared__ __attribute__((aligned(16))) float lds[kFpLds];
    __shared__ float weights[kMask ? 256 : 1];
    const int tid = threadIdx.x;
    const int group = blockIdx.x % a.groups, slice0 = blockIdx.x / a.groups * (R * T);
    const ForwardView* __restrict__ views = a.views;
    const int nu = a.nu, nv = a.nv, zdir = a.zdir, band = a.band;
    const int row0 = group * P, rows = min(P, nv - row0);
    const int nx = s.res[0], nz = s.res[2];
    const int columns = nu << a.shift;       // ray columns of a projection
    const float sd = 1.0f / (float)a.sub, off = sd / 2.0f;
    if constexpr (kMask) {
        for (int i = tid; i < 256; i += T) weights[i] = (float)i / 255.0f;
        __syncthreads();
    }
    // the planes of the rows, the same for every projection (checked on the host)
    int plane[P];
    bool hit[P];
    bool any = false;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const ForwardView& f = views[0];
        const float fy = (float)min(row0 + p, nv - 1) + off;
        const float ru = f.h[1] * off, rv = f.v[1] * fy;
        const float src = f.source[1] + ru + rv;
        const float t0 = (s.bmin[1] - src) * -FLT_MAX, t1 = (s.bmax[1] - src) * -FLT_MAX;
        hit[p] = p < rows && fminf(t0, t1) < 0.0f && fmaxf(t0, t1) > 0.0f;
        const float y = fminf(fmaxf(src, s.bmin[1]), s.bmax[1]);
        plane[p] = min(max((int)((y - s.bmin[1]) * (1.0f / s.vs[1])), 0), s.res[1] - 1);
        any = any || hit[p];
    }

    // ray column of slot r: false where there is none
    auto column = [&](int r, int& q, int& u, int& si) {
        const int id = slice0 + r * T + tid;
        q = id / columns;
        const int rem = id - q * columns;
        u = rem >> a.shift;
        si = rem & ((1 << a.shift) - 1);
        return q < a.n && si < a.sub;
    };
    SweepRay<kMask, P> ray[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        SweepRay<kMask, P>& y = ray[r];
        y.left = 0;
        y.at = 0;
        y.rx = y.rz = y.stepx = y.stepz = 0.0f;
        y.dx = y.dz = 0;
#pragma unroll
        for (int p = 0; p < P; ++p) y.acc[p] = 0.0f;
#pragma unroll
        for (int p = 0; p < (kMask ? P : 1); ++p) y.len[p] = 0.0f;
        int q, u, si;
        if (column(r, q, u, si) && any) {
            const ForwardView& f = views[q];
            RayParams g;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                g.source[k] = f.source[k];
                g.h[k] = f.h[k];
                g.v[k] = f.v[k];
                g.ray[k] = f.ray[k];
            }
            const DdaConst c = dda_const(g.ray, s.vs);
            float src[3];
            fp_ray_source(g, (uint32_t)u, (uint32_t)row0, (uint32_t)si, 0, sd, off, src);
            SlabParams flat = s;
            src[1] = 0.0f;
            flat.bmin[1] = -1.0f;
            flat.bmax[1] = 1.0f;
            DdaRay d;
            dda_begin(flat, c, src, d);
            y.rx = d.res[0];
            y.rz = d.res[2];
            y.stepx = c.step[0];
            y.stepz = c.step[2];
            y.at = (d.vox[2] * nx + d.vox[0]) * W * 4;
            y.left = !d.live ? 0 : c.sign[0] > 0 ? nx - d.vox[0] : c.sign[0] < 0 ? d.vox[0] + 1 : 0x7fffffff;
            y.dx = c.sign[0] * W * 4;
            y.dz = c.sign[2] * nx * W * 4;
        }
    }

    if (any) {
        const size_t slice = (size_t)s.nx * s.ny;
        const typename S::T* base[P];
        const uint8_t* mbase[P];
#pragma unroll
        for (int p = 0; p < P; ++p) {
            base[p] = vol + s.first_voxel + (size_t)plane[p] * s.nx;
            if constexpr (kMask) mbase[p] = a.mask + s.first_voxel + (size_t)plane[p] * s.nx;
        }
        const int bands = (nz + band - 1) / band;
        // items of G voxels in x, P planes each: the next band's are in flight
        // while the rays cross this one
        constexpr int G = kVec ? 4 : 1, kItems = kFpLds / (G * W * T);
        const int items_x = nx / G;
        typename std::conditional<kVec, typename Q::V, typename S::T>::type pre[kItems][P];
        typename std::conditional<kVec, uint32_t, uint8_t>::type mpre[kMask ? kItems : 1][P];
        auto range = [&](int b, int& z0, int& z1) {
            z0 = (zdir >= 0 ? b : bands - 1 - b) * band;
            z1 = min(z0 + band, nz);
        };
        // item k T + tid of a band: its offset follows from the one before it (a
        // band's offsets fit 32 bits: the host checks it)
        const int first_z = tid / items_x, first_x = tid - first_z * items_x;
        const uint32_t offset0 = (uint32_t)first_z * (uint32_t)slice + (uint32_t)(first_x * G);
        const int next_x = T % items_x;
        const uint32_t next = (uint32_t)(T / items_x) * (uint32_t)slice + (uint32_t)(next_x * G);
        const uint32_t wrap = (uint32_t)slice - (uint32_t)nx;
        auto load = [&](int z0, int z1) {
            const uint32_t last = (uint32_t)(z1 - z0 - 1) * (uint32_t)slice + (uint32_t)(nx - G);
            uint32_t offset = offset0;
            int x = first_x;
#pragma unroll
            for (int k = 0; k < kItems; ++k) {
                const uint32_t at = min(offset, last);   // (beyond the band: read again, not used)
#pragma unroll
                for (int p = 0; p < P; ++p) {
                    const typename S::T* from = base[p] + (size_t)z0 * slice;
                    if constexpr (kVec) pre[k][p] = *reinterpret_cast<const typename Q::V*>(from + at);
                    else pre[k][p] = from[at];
                    if constexpr (kMask) {
                        const uint8_t* mfrom = mbase[p] + (size_t)z0 * slice;
                        if constexpr (kVec) mpre[k][p] = *reinterpret_cast<const uint32_t*>(mfrom + at);
                        else mpre[k][p] = mfrom[at];
                    }
                }
                x += next_x;
                offset += next;
                if (x >= items_x) {
                    x -= items_x;
                    offset += wrap;
                }
            }
        };
        int z0, z1;
        range(0, z0, z1);
        load(z0, z1);
        for (int b = 0; b < bands; ++b) {
            range(b, z0, z1);
            const int m = (z1 - z0) * items_x;
#pragma unroll
            for (int k = 0; k < kItems; ++k) {
                const int i = k * T + tid;
                if (i < m) {
                    if constexpr (kVec) {
                        float v[W][4];
#pragma unroll
                        for (int p = 0; p < P; ++p) {
                            Q::unpack(pre[k][p], v[p]);
                            if constexpr (kMask)
#pragma unroll
                                for (int j = 0; j < 4; ++j) v[P + p][j] = weights[mpre[k][p] >> (8 * j) & 255u];
                        }
                        interleave<W>(v, reinterpret_cast<f32x4*>(lds) + (size_t)i * W);
                    } else {
                        typename L::V cell;
                        float* to = reinterpret_cast<float*>(&cell);
#pragma unroll
                        for (int p = 0; p < P; ++p) {
                            to[p] = S::load(&pre[k][p], 0);
                            if constexpr (kMask) to[P + p] = weights[mpre[k][p]];
                        }
                        reinterpret_cast<typename L::V*>(lds)[i] = cell;
                    }
                }
            }
            if (b + 1 < bands) {
                int n0, n1;
                range(b + 1, n0, n1);
                load(n0, n1);
            }
            __syncthreads();
            const unsigned bytes = (unsigned)((z1 - z0) * nx * W) * 4u;
            const int start = z0 * nx * W * 4;
            const char* rows_at = reinterpret_cast<const char*>(lds);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                SweepRay<kMask, P>& y = ray[r];
                int at = y.at - start, left = y.left;
                float rx = y.rx, rz = y.rz;
                while (left != 0 && (unsigned)at < bytes) {
                    const typename L::V v = *reinterpret_cast<const typename L::V*>(rows_at + at);
                    const bool ix = rx <= rz;
                    const float dt = ix ? rx : rz, rest = fabsf(rx - rz);
                    rx = ix ? y.stepx : rest;
                    rz = ix ? rest : y.stepz;
                    at += ix ? y.dx : y.dz;
                    left -= ix ? 1 : 0;
#pragma unroll
                    for (int p = 0; p < P; ++p) y.acc[p] = fmaf(dt, L::get(v, p), y.acc[p]);
                    if constexpr (kMask) {
#pragma unroll
                        for (int p = 0; p < P; ++p) y.len[p] = fmaf(dt, L::get(v, P + p), y.len[p]);
                    } else {
                        y.len[0] += dt;
                    }
                }
                y.at = at + start;
                y.left = left;
                y.rx = rx;
                y.rz = rz;
            }
            __syncthreads();
        }
    }

#pragma unroll
    for (int r = 0; r < R; ++r) {
        int q, u, si;
        const bool mine = column(r, q, u, si) && si == 0;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            // the pixel's sub-rays in the fused kernels' order: those of a column
            // differ only in y and have equal sums
            float acc = 0.0f, len = 0.0f;
            const float ra = hit[p] ? ray[r].acc[p] : 0.0f, rl = hit[p] ? ray[r].len[kMask ? p : 0] : 0.0f;
            for (int k = 0; k < a.sub; ++k) {
                const float ka = a.sub > 1 ? __shfl_down(ra, k) : ra, kl = a.sub > 1 ? __shfl_down(rl, k) : rl;
                for (int j = 0; j < a.sub; ++j) {
                    acc += ka;
                    len += kl;
                }
            }
            if (!mine || p >= rows) continue;
            const ForwardView& f = views[q];
            const size_t i = (size_t)(row0 + p) * nu + u;
            const float total = (float)(a.sub * a.sub);
            float pv = 0.0f + acc / total, l = 0.0f + len / total;
            if (f.use_loc) {
                pv = l > kEpsilon ? pv * f.loc_c / l : 0.0f;
                l = f.loc_c;
            }
            if (f.raw) {
                f.residual[i] = pv;
                f.length[i] = l;
                continue;
            }
            float b;
            if (f.measured_type == ETN_VOXEL_FLOAT16) b = F16::load(static_cast<const __half*>(f.measured), i);
            else if (f.measured_type == ETN_VOXEL_BFLOAT16) b = BF16::load(static_cast<const uint16_t*>(f.measured), i);
            else b = static_cast<const float*>(f.measured)[i];
            f.residual[i] = b - pv;
            f.length[i] = l;
        }
    }
}

template <typename S, bool kVec, bool kMask, int P>
void launch_sweep_forward(const SlabParams& s, SweepForward a, const ForwardShape& shape, const void* volume,
                          hipStream_t stream)
{
    constexpr int T = kFpThreads;
    const auto* vol = static_cast<const typename S::T*>(volume);
    a.groups = (a.nv + P - 1) / P;
    a.band = std::max(1, std::min(s.res[2], kFpLds / (s.res[0] * P * (kMask ? 2 : 1))));
    auto launch = [&](auto kernel) { kernel<<<(unsigned)shape.workgroups, T, 0, stream>>>(s, a, vol); };
    const int rays = shape.rays;
    if (rays == 1) launch(sweep_forward_kernel<S, kVec, kMask, P, 1>);
    else if (rays == 2) launch(sweep_forward_kernel<S, kVec, kMask, P, 2>);
    else if (rays == 4) launch(sweep_forward_kernel<S, kVec, kMask, P, 4>);
    else launch(sweep_forward_kernel<S, kVec, kMask, P, 8>);
}

template <typename S, bool kMask>
void sweep_forward_typed(const SlabParams& s, const SweepForward& a, const void* volume, hipStream_t stream)
{
    const bool vec = s.res[0] % 4 == 0 && reinterpret_cast<uintptr_t>(volume) % (4 * sizeof(typename S::T)) == 0 &&
                     reinterpret_cast<uintptr_t>(a.mask) % 4 == 0;
    const ForwardShape shape = sweep_forward_shape(s.res[0], a.n, (uint32_t)a.nu, (uint32_t)a.nv, a.sub, kMask);
    auto launch = [&](auto v) {
        constexpr bool kVec = decltype(v)::value;
        if constexpr (!kMask) {
            if (shape.planes == 4) return launch_sweep_forward<S, kVec, kMask, 4>(s, a, shape, volume, stream);
        }
        if (shape.planes == 2) launch_sweep_forward<S, kVec, kMask, 2>(s, a, shape, volume, stream);
        else launch_sweep_forward<S, kVec, kMask, 1>(s, a, shape, volume, stream);
    };
    if (vec) launch(std::true_type{});
    else launch(std::false_type{});
}

// ---- oversampled and masked back projections in one sweep -------------------------
// The fused kernels' fast arithmetic, operation for operation and in their sample
// order: with kOver the per_dir x per_dir pattern (PD = per_dir) of their sample
// loop, without it their single-sample update with a mask weight (PD = 1).  A
// sample's u does not depend on its pattern row, which only moves it along y, nor
// on the plane: the columns and weights of a pattern row's PD samples are worked
// out once for all PD rows of all four planes, so a sample costs its record read
// and 10 instruction slots (19 on the fused kernels, which also leave CUs idle
// where the planes are no multiple of them).  A workgroup owns four planes x 64
// columns x 4 kSampleDepth slices in registers.  250 x 300 x 150 bf16 with a mask,
// 3 x 3 samples: 0.068 ms, with the forward sweep 0.110 where a fused pass takes
// 0.25 (0.052 with a pattern row's contributions added before their weight, a
// different rounding).
constexpr int kSampleDepth = 4;      // slices a wave

template <typename S, int PD, bool kOver>
__global__ void __launch_bounds__(kSweepThreads, 4)
    sweep_samples_kernel(SlabParams s, const SampleView* __restrict__ views, int n, typename S::T* vol,
                         const uint8_t* __restrict__ mask, int nu, int nv)
{
    constexpr int kPlanes = PD >= 3 ? 2 : kSweepPlanes;   // planes whose reads are in flight together
    __shared__ f32x4 recs[kSweepPlanes * PD][kSweepColumns];
    __shared__ float weights[256];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int x0 = blockIdx.x * kSweepTile, y0 = blockIdx.y * kSweepPlanes, z0 = blockIdx.z * (4 * kSampleDepth);
    const int x = x0 + lane, zw = z0 + wave * kSampleDepth;
    const int planes = min(kSweepPlanes, s.res[1] - y0);
    const bool xin = x < s.res[0];
    const size_t slice = (size_t)s.nx * s.ny;
    const size_t at0 = s.first_voxel + (size_t)zw * slice + (size_t)y0 * s.nx + (size_t)(uint32_t)x;
    weights[tid] = (float)tid / 255.0f;

    // (addresses are clamped into the volume: nothing waits for a single load)
    float value[kSampleDepth][kSweepPlanes];
    uint32_t mv[kSampleDepth];
    auto clamped = [&](int j, int p) {
        return s.first_voxel + (size_t)min(zw + j, s.res[2] - 1) * slice + (size_t)(y0 + min(p, planes - 1)) * s.nx +
               (size_t)min(x, s.res[0] - 1);
    };
#pragma unroll
    for (int j = 0; j < kSampleDepth; ++j)
#pragma unroll
        for (int p = 0; p < kSweepPlanes; ++p) value[j][p] = S::load(vol, clamped(j, p));
    if (mask) {
        uint32_t in[kSampleDepth][kSweepPlanes];
#pragma unroll
        for (int j = 0; j < kSampleDepth; ++j)
#pragma unroll
            for (int p = 0; p < kSweepPlanes; ++p) in[j][p] = mask[clamped(j, p)];
#pragma unroll
        for (int j = 0; j < kSampleDepth; ++j) mv[j] = in[j][0] | in[j][1] << 8 | in[j][2] << 16 | in[j][3] << 24;
    } else {
#pragma unroll
        for (int j = 0; j < kSampleDepth; ++j) mv[j] = 0xffffffffu;
    }
    const float xc = s.bmin[0] + ((float)x + 0.5f) * s.vs[0];
    // the tile's corners
    const float cxa = s.bmin[0] + ((float)x0 + 0.5f) * s.vs[0], cxb = s.bmin[0] + ((float)(x0 + kSweepTile - 1) + 0.5f) * s.vs[0];
    const float cza = s.bmin[2] + ((float)z0 + 0.5f) * s.vs[2];
    const float czb = s.bmin[2] + ((float)(z0 + 4 * kSampleDepth - 1) + 0.5f) * s.vs[2];

    for (int q = 0; q < n; ++q) {
        const SampleView& v = views[q];
        const float m0 = v.m0, m8 = v.m8, m12 = v.m12;
        // the tile's smallest u, less one for its rounding
        float sxa = v.sx[0], sxb = v.sx[0], sza = v.sz[0], szb = v.sz[0];
#pragma unroll
        for (int i = 1; i < PD; ++i) {
            sxa = fminf(sxa, v.sx[i]);
            sxb = fmaxf(sxb, v.sx[i]);
            sza = fminf(sza, v.sz[i]);
            szb = fmaxf(szb, v.sz[i]);
        }
        const float umin = (m0 >= 0.0f ? m0 * (cxa + sxa) : m0 * (cxb + sxb)) +
                           (m8 >= 0.0f ? m8 * (cza + sza) : m8 * (czb + szb)) + m12 - 0.5f;
        const int first = (int)floorf(umin) - 1;
        __syncthreads();
        // records {A, B, LA, LB} of a plane's pattern rows: R = A + B tx, L = LA + LB
        // tx.  Thread (h, k) takes column k of rows h, h + 2, ...; the loads of PD of
        // them are in flight together (clamped into the images, what lies outside
        // zeroed afterwards)
        const int k = tid % kSweepColumns, h = tid / kSweepColumns, u0 = first + k;
        const bool c0 = (unsigned)u0 < (unsigned)nu, c1 = (unsigned)(u0 + 1) < (unsigned)nu;
        const uint32_t k0 = (uint32_t)min(max(u0, 0), nu - 1), k1 = (uint32_t)min(max(u0 + 1, 0), nu - 1);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            float in[PD][8], ty[PD];
            int r0[PD];
#pragma unroll
            for (int e = 0; e < PD; ++e) {
                const int row = (half * PD + e) * 2 + h, p = row / PD;
                const float py = s.bmin[1] + ((float)(y0 + p) + 0.5f) * s.vs[1];
                float vp = v.m5 * (py + v.sy[row - p * PD]);
                vp = vp + v.m13 * 1.0f;
                float base_row;
                ty[e] = cl_fract(vp - 0.5f, &base_row);
                r0[e] = __builtin_amdgcn_readfirstlane((int)base_row);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const size_t at = (size_t)min(max(r0[e] + i, 0), nv - 1) * nu;
                    in[e][2 * i] = (v.residual + at)[k0];
                    in[e][2 * i + 1] = (v.residual + at)[k1];
                    in[e][4 + 2 * i] = (v.length + at)[k0];
                    in[e][5 + 2 * i] = (v.length + at)[k1];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < PD; ++e) {
                float w[8];
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const bool rin = (unsigned)(r0[e] + (t >> 1 & 1)) < (unsigned)nv;
                    w[t] = (rin & (t & 1 ? c1 : c0)) ? in[e][t] : 0.0f;
                }
                const float dr0 = w[1] - w[0], dr1 = w[3] - w[2], dl0 = w[5] - w[4], dl1 = w[7] - w[6];
                // (a single sample's A and B carry lambda times the chord)
                const float lc = kOver ? 1.0f : v.lambda * v.sw[0];
                recs[(half * PD + e) * 2 + h][k] = f32x4{lc * fmaf(w[2] - w[0], ty[e], w[0]), lc * fmaf(dr1 - dr0, ty[e], dr0),
                                                         fmaf(w[6] - w[4], ty[e], w[4]), fmaf(dl1 - dl0, ty[e], dl0)};
            }
        }
        __syncthreads();
        const f32x4* rec = recs[0] - first;
#pragma unroll
        for (int j = 0; j < kSampleDepth; ++j) {
            const float zc = s.bmin[2] + ((float)(zw + j) + 0.5f) * s.vs[2];
            // the columns and weights of a pattern row's samples
            const f32x4* at[PD];
            float tx[PD];
#pragma unroll
            for (int i = 0; i < PD; ++i) {
                float u = m0 * (xc + v.sx[i]) + 0.0f;
                u = u + m8 * (zc + v.sz[i]);
                u = u + m12 * 1.0f;
                u = u - 0.5f;
                int column;
                if constexpr (kOver) {
                    const float base = floorf(u);
                    tx[i] = u - base;
                    column = (int)base;
                } else {
                    tx[i] = __builtin_amdgcn_fractf(u);
                    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(column) : "v"(u));
                }
                at[i] = rec + column;
            }
            if constexpr (kOver) {
                float sum[kSweepPlanes];
                int used[kSweepPlanes];
#pragma unroll
                for (int p = 0; p < kSweepPlanes; ++p) {
                    sum[p] = 0.0f;
                    used[p] = 0;
                }
#pragma unroll 1
                for (int ys = 0; ys < PD; ++ys) {
#pragma unroll
                    for (int p0 = 0; p0 < kSweepPlanes; p0 += kPlanes) {
                        float R[PD][kPlanes], L[PD][kPlanes], least = FLT_MAX;
#pragma unroll
                        for (int i = 0; i < PD; ++i)
#pragma unroll
                            for (int p = 0; p < kPlanes; ++p) {
                                const f32x4 e = at[i][((p0 + p) * PD + ys) * kSweepColumns];
                                R[i][p] = fmaf(e[1], tx[i], e[0]);
                                L[i][p] = fmaf(e[3], tx[i], e[2]);
                                least = __builtin_elementwise_minimum(least, L[i][p]);   // (a NaN stays)
                            }
                        // the common case, every record with rays through it, decided for
                        // the whole wave: no test, count or select a sample
                        const bool all = __all(least > kEpsilon);
#pragma unroll
                        for (int p = 0; p < kPlanes; ++p) used[p0 + p] += all ? PD : 0;
#pragma unroll
                        for (int i = 0; i < PD; ++i) {
                            const float lw = v.lambda * v.sw[i];
#pragma unroll
                            for (int p = 0; p < kPlanes; ++p) {
                                const float contrib = R[i][p] * lw * __builtin_amdgcn_rcpf(L[i][p]);
                                if (all) {
                                    sum[p0 + p] += contrib;
                                } else {
                                    const bool ok = L[i][p] > kEpsilon;
                                    sum[p0 + p] += ok ? contrib : 0.0f;
                                    used[p0 + p] += ok ? 1 : 0;
                                }
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
#pragma unroll
                for (int p = 0; p < kSweepPlanes; ++p) {
                    if (used[p] != 0) value[j][p] += weights[mv[j] >> (8 * p) & 255u] * sum[p] / (float)used[p];
                }
            } else {
#pragma unroll
                for (int p = 0; p < kSweepPlanes; ++p) {
                    const f32x4 e = at[0][p * kSweepColumns];
                    const float R = fmaf(e[1], tx[0], e[0]), L = fmaf(e[3], tx[0], e[2]);
                    const float next = fmaf(weights[mv[j] >> (8 * p) & 255u], R * __builtin_amdgcn_rcpf(L), value[j][p]);
                    value[j][p] = L > kEpsilon ? next : value[j][p];
                }
            }
            round_planes<S>(value[j]);
        }
    }
#pragma unroll
    for (int j = 0; j < kSampleDepth; ++j)
#pragma unroll
        for (int p = 0; p < kSweepPlanes; ++p)
            if (zw + j < s.res[2] && p < planes && xin)
                S::store(vol, at0 + (size_t)j * slice + (size_t)p * s.nx, value[j][p]);
}

template <typename S>
void sweep_samples_typed(const SlabParams& s, const SampleView* views, int n, int per_dir, bool over, uint32_t nu,
                         uint32_t nv, void* volume, const uint8_t* mask, hipStream_t stream)
{
    auto* vol = static_cast<typename S::T*>(volume);
    const dim3 grid((s.res[0] + kSweepTile - 1) / kSweepTile, (s.res[1] + kSweepPlanes - 1) / kSweepPlanes,
                    (s.res[2] + 4 * kSampleDepth - 1) / (4 * kSampleDepth));
    auto launch = [&](auto kernel) {
        kernel<<<grid, kSweepThreads, 0, stream>>>(s, views, n, vol, mask, (int)nu, (int)nv);
    };
    if (!over) launch(sweep_samples_kernel<S, 1, false>);
    else if (per_dir == 1) launch(sweep_samples_kernel<S, 1, true>);
    else if (per_dir == 2) launch(sweep_samples_kernel<S, 2, true>);
    else if (per_dir == 3) launch(sweep_samples_kernel<S, 3, true>);
    else launch(sweep_samples_kernel<S, 4, true>);
}

}  // namespace

bool plane_forward_project(const SlabParams& s, const RayParams& r, etn_voxel_type vt, const void* volume,
                           float* projection, float* traversal_length, hipStream_t stream)
{
    if (!plane_forward_fits(s, r)) return false;
    // A row's whole plane is staged however few rays cross it: us for the planes
    // (less a voxel where several rows share one) and for one ray after another's
    // steps on the generic kernel, which also slows down with the rays in flight.
    // Staged / generic: 1000^3 10 columns 590 / 521, 32 columns 590 / 653; 850^3
    // (single voxels) 64 columns 687 / 582, 128 columns 691 / 665; 1000 x 128 x 1000
    // 128 columns x 2048 rows 838 / 571; 700^3 10 columns 254 / 358
    const size_t voxel = vt == ETN_VOXEL_FLOAT32 ? 4 : 2;
    const double rate = !vector_rows(s, volume, voxel) ? 1.12e-6
                        : r.nv >= 2u * (uint32_t)s.res[1] ? 0.42e-6
                        : voxel == 4 ? 0.59e-6 : 0.36e-6;
    const double staged = rate * r.nv * s.res[0] * s.res[2];
    const double rays = (double)r.nu * std::min(r.nv, (uint32_t)s.res[1]);
    if (staged > 0.25 * (s.res[0] + s.res[2]) * (1.0 + rays * 1e-5)) return false;
    if (vt == ETN_VOXEL_FLOAT16) launch_forward_typed<F16>(s, r, volume, projection, traversal_length, stream);
    else if (vt == ETN_VOXEL_BFLOAT16) launch_forward_typed<BF16>(s, r, volume, projection, traversal_length, stream);
    else launch_forward_typed<F32>(s, r, volume, projection, traversal_length, stream);
    hip_check(hipGetLastError(), "forward projection launch");
    return true;
}

bool plane_back_project(const SlabParams& s, const BpParams& b, etn_voxel_type vt, void* volume, const float* residual,
                        const float* ray_length, hipStream_t stream)
{
    const BackTile t = plane_back_tile(s, b);
    if (t.depth == 0) return false;
    const dim3 grid((s.res[0] + (1 << t.shift) - 1) >> t.shift, (s.res[1] + kBpPlanes - 1) / kBpPlanes,
                    (s.res[2] + t.depth - 1) / t.depth);
    auto launch = [&](auto type) {
        using S = decltype(type);
        plane_back_kernel<S><<<grid, kBpThreads, 0, stream>>>(s, b, static_cast<typename S::T*>(volume), residual,
                                                              ray_length, t.depth, t.shift);
    };
    if (vt == ETN_VOXEL_FLOAT16) launch(F16{});
    else if (vt == ETN_VOXEL_BFLOAT16) launch(BF16{});
    else launch(F32{});
    hip_check(hipGetLastError(), "back projection launch");
    return true;
}

bool make_back_view(const SlabParams& s, const BpParams& b, const float* residual, const float* length, BackView* out)
{
    if (b.nsamples != 1 || !single_axis_matrix(s, b)) return false;
    const float* m = b.m;
    const float columns = (std::fabs(m[0]) * s.vs[0] + std::fabs(m[8]) * s.vs[2]) * (float)(kSweepTile - 1) + 5.0f;
    if (!(columns <= (float)kSweepColumns)) return false;
    if ((s.res[1] + kSweepPlanes - 1) / kSweepPlanes > 65535 || (s.res[2] + kSweepTile - 1) / kSweepTile > 65535)
        return false;
    if ((uint64_t)b.nu * b.nv > 0x3fffffffu) return false;   // image offsets in 32-bit bytes
    const float4 e = b.samples[0];
    *out = {m[0], m[8], m[12], m[5], m[13], e.x, e.y, e.z, b.lambda * e.w, residual, length};
    return true;
}

SweepGroups sweep_groups(const SlabParams& s, const BackView* views, int n, uint32_t nv,
                         const std::vector<uint8_t>& row_class)
{
    // whether the planes of a group read rows of equal lengths (the kernel's own
    // arithmetic for the row of a plane)
    auto equal = [&](int group) {
        const BackView& v = views[0];
        for (int p = 0; p < kSweepPlanes && group * kSweepPlanes + p < s.res[1]; ++p) {
            const float py = s.bmin[1] + ((float)(group * kSweepPlanes + p) + 0.5f) * s.vs[1];
            float vp = v.m5 * (py + v.sy);
            vp = vp + v.m13 * 1.0f;
            const int row = (int)std::floor(vp - 0.5f);
            for (int r = row; r <= row + 1; ++r)
                if (r < 0 || r >= (int)nv || row_class[r] == 0) return false;
        }
        return true;
    };
    SweepGroups g;
    // every projection reads a plane's rows with the same weights
    for (int q = 1; q < n; ++q)
        if (views[q].m5 != views[0].m5 || views[q].m13 != views[0].m13 || views[q].sy != views[0].sy) return g;
    g.count = (s.res[1] + kSweepPlanes - 1) / kSweepPlanes;
    // the longest run of such groups
    for (int i = 0; i < g.count;) {
        int e = i;
        while (e < g.count && equal(e)) ++e;
        if (e - i > g.end - g.begin) {
            g.begin = i;
            g.end = e;
        }
        i = std::max(e, i) + 1;
    }
    return g;
}

namespace {
template <typename S>
void sweep_back_typed(const SlabParams& s, const SweepGroups& g, const BackView* views, int n, uint32_t nu, uint32_t nv,
                      void* volume, hipStream_t stream)
{
    auto* vol = static_cast<typename S::T*>(volume);
    const dim3 grid((s.res[0] + kSweepTile - 1) / kSweepTile, g.count, (s.res[2] + kSweepTile - 1) / kSweepTile);
    sweep_back_kernel<S><<<grid, kSweepThreads, 0, stream>>>(s, views, n, vol, (int)nu, (int)nv, g.begin, g.end);
}
}  // namespace

void sweep_back_project(const SlabParams& s, const SweepGroups& g, const BackView* views, int n, uint32_t nu,
                        uint32_t nv, etn_voxel_type vt, void* volume, hipStream_t stream)
{
    if (n <= 0) return;
    if (vt == ETN_VOXEL_FLOAT16) sweep_back_typed<F16>(s, g, views, n, nu, nv, volume, stream);
    else if (vt == ETN_VOXEL_BFLOAT16) sweep_back_typed<BF16>(s, g, views, n, nu, nv, volume, stream);
    else sweep_back_typed<F32>(s, g, views, n, nu, nv, volume, stream);
    hip_check(hipGetLastError(), "back projection sweep launch");
}

bool forward_view_fits(const SlabParams& s, const ForwardView& v, uint32_t nu, uint32_t nv, int sub, bool masked)
{
    RayParams r{};
    for (int k = 0; k < 3; ++k) {
        r.source[k] = v.source[k];
        r.h[k] = v.h[k];
        r.v[k] = v.v[k];
        r.ray[k] = v.ray[k];
    }
    r.nu = nu;
    r.nv = nv;
    r.samples = 1;
    if (sub < 1 || sub > 4 || nu > 1u << 20 || nv > 1u << 20 || s.res[1] > 65535) return false;
    return s.res[0] * (masked ? 2 : 1) <= kFpLds && plane_geometry_fits(s, r, sub);
}

ForwardShape sweep_forward_shape(int nx, int n, uint32_t nu, uint32_t nv, int sub, bool masked)
{
    int shift = 0;
    while (1 << shift < sub) ++shift;
    const int columns = n * (int)(nu << shift), w = masked ? 2 : 1;
    auto groups = [&](int planes) { return ((int)nv + planes - 1) / planes; };
    auto slices = [&](int rays) { return (columns + rays * kFpThreads - 1) / (rays * kFpThreads); };
    // planes a workgroup: four where they and the columns still make a
    // workgroup for every CU (two planes: 240 us), fewer on small volumes; a
    // voxel's values and weights are one 16-byte read
    auto fills = [&](int planes) { return nx * planes * w <= kFpLds && groups(planes) * slices(1) >= 256; };
    ForwardShape f{!masked && fills(4) ? 4 : fills(2) ? 2 : 1, 8, 0};
    // columns a thread: as many as there are, fewer where that leaves a CU fewer
    // than two workgroups (512 x 512 x 256, eight projections: 167 us a sweep
    // with two a CU, 175 with one)
    while (f.rays > 1 && (f.rays / 2 * kFpThreads >= columns || groups(f.planes) * slices(f.rays) < 512)) f.rays /= 2;
    f.workgroups = groups(f.planes) * slices(f.rays);
    return f;
}

void sweep_forward_project(const SlabParams& s, const ForwardView* views, int n, int zdir, uint32_t nu, uint32_t nv,
                           int sub, etn_voxel_type vt, const void* volume, const uint8_t* mask, hipStream_t stream)
{
    if (n <= 0) return;
    if (n > kSweepForward) fail("forward projection sweep: at most eight projections");
    SweepForward a{};
    a.views = views;
    a.n = n;
    a.zdir = zdir;
    a.nu = (int)nu;
    a.nv = (int)nv;
    a.sub = sub;
    while (1 << a.shift < sub) ++a.shift;
    a.mask = mask;
    auto launch = [&](auto type) {
        using S = decltype(type);
        if (mask) sweep_forward_typed<S, true>(s, a, volume, stream);
        else sweep_forward_typed<S, false>(s, a, volume, stream);
    };
    if (vt == ETN_VOXEL_FLOAT16) launch(F16{});
    else if (vt == ETN_VOXEL_BFLOAT16) launch(BF16{});
    else launch(F32{});
    hip_check(hipGetLastError(), "forward projection sweep launch");
}

bool make_sample_view(const SlabParams& s, const BpParams& b, const float* residual, const float* length, SampleView* out)
{
    int pd = 1;
    while (pd * pd < (int)b.nsamples) ++pd;
    if (pd > 4 || pd * pd != (int)b.nsamples || !single_axis_matrix(s, b)) return false;
    const float* m = b.m;
    SampleView v{m[0], m[8], m[12], m[5], m[13], b.lambda, {}, {}, {}, {}, residual, length};
    for (int t = 0; t < pd * pd; ++t) {
        const float4 e = b.samples[t];
        const int ys = t / pd, i = t - ys * pd;
        if (i == 0) v.sy[ys] = e.y;
        if (ys == 0) {
            v.sx[i] = e.x;
            v.sz[i] = e.z;
            v.sw[i] = e.w;
        }
        // a pattern row only moves its samples along y
        if (v.sy[ys] != e.y || v.sx[i] != e.x || v.sz[i] != e.z || v.sw[i] != e.w) return false;
    }
    const float spread = std::fabs(m[0]) * (*std::max_element(v.sx, v.sx + pd) - *std::min_element(v.sx, v.sx + pd)) +
                         std::fabs(m[8]) * (*std::max_element(v.sz, v.sz + pd) - *std::min_element(v.sz, v.sz + pd));
    const float columns = std::fabs(m[0]) * s.vs[0] * (float)(kSweepTile - 1) +
                          std::fabs(m[8]) * s.vs[2] * (float)(4 * kSampleDepth - 1) + spread + 5.0f;
    if (!(columns <= (float)kSweepColumns)) return false;
    if ((s.res[1] + kSweepPlanes - 1) / kSweepPlanes > 65535 || s.res[2] / (4 * kSampleDepth) >= 65535) return false;
    *out = v;
    return true;
}

void sweep_samples_project(const SlabParams& s, const SampleView* views, int n, int per_dir, bool over, uint32_t nu,
                           uint32_t nv, etn_voxel_type vt, void* volume, const uint8_t* mask, hipStream_t stream)
{
    if (n <= 0) return;
    if (!over && per_dir != 1) fail("back projection sweep: a sample pattern is oversampled");
    if (vt == ETN_VOXEL_FLOAT16) sweep_samples_typed<F16>(s, views, n, per_dir, over, nu, nv, volume, mask, stream);
    else if (vt == ETN_VOXEL_BFLOAT16) sweep_samples_typed<BF16>(s, views, n, per_dir, over, nu, nv, volume, mask, stream);
    else sweep_samples_typed<F32>(s, views, n, per_dir, over, nu, nv, volume, mask, stream);
    hip_check(hipGetLastError(), "back projection sweep launch");
}

std::vector<uint8_t> row_classes(const SlabParams& s, const RayParams& r)
{
    std::vector<uint8_t> out(r.nv, 0);
    if (r.ray[1] != 0.0f || r.h[1] != 0.0f || r.v[0] != 0.0f || r.v[2] != 0.0f) return out;
    for (uint32_t y = 0; y < r.nv; ++y) {
        const float fy = (float)y + 0.5f;
        const float rv = r.v[1] * fy;
        const float src = r.source[1] + 0.0f + rv;
        const float t0 = (s.bmin[1] - src) * -FLT_MAX, t1 = (s.bmax[1] - src) * -FLT_MAX;
        out[y] = std::fmin(t0, t1) < -1e30f && std::fmax(t0, t1) > 1e30f ? 1 : 0;
    }
    return out;
}

}  // namespace dev
}  // namespace etn
