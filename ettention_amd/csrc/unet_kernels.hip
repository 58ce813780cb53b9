// Learned correction network kernels (see unet_kernels.hpp).
//
// The 3x3x3 convolution is an implicit GEMM on the matrix cores: output
// voxels are the GEMM rows, output channels the columns, and the reduction
// runs over k = tap * cin + ci.  Each wave owns MT tiles of 16 voxels and all
// cout channels (NT tiles of 16); per 32-wide k step a lane loads its 8
// channels of one tap for each voxel tile (one 16-byte load from the
// channels-last activation, or zeros outside the volume) and 8 weights per
// channel tile, then issues MT x NT v_mfma_f32_16x16x32_bf16.  Lane layouts
// (checked on the device): A[i][k] in lane i + 16 (k / 8), element k % 8;
// B[k][j] in lane j + 16 (k / 8); D[i][j] in lane j + 16 (i / 4), element i % 4.
//
// The weight gradient is the GEMM dW[co][(tap, ci)] = sum_m gy[m][co] x[m + d(tap)][ci]
// with the voxels as the reduction, over LDS-staged bricks read transposed
// (conv3_wgrad_kernel); the workgroups' partial sums are added in a fixed
// order, so every gradient is deterministic.
#include <algorithm>

#include "common.hpp"
#include "device_math.hpp"
#include "unet_kernels.hpp"

namespace etn {
namespace nn {

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ uint16_t f2bf(float f) { return dev::BF16::pack(f); }

__device__ __forceinline__ u32x4 load16(const uint16_t* p) { return *reinterpret_cast<const u32x4*>(p); }
__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

constexpr int kConvWaves = 4;
constexpr int kThreads = 256;

// ---- 3x3x3 convolution, implicit GEMM ---------------------------------------
template <int NT, int MT>
__global__ void __launch_bounds__(kThreads) conv3_fwd_kernel(ConvArgs a)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane & 15, kg = lane >> 4;
    const size_t M = (size_t)a.D * a.H * a.W;
    const size_t m0 = ((size_t)blockIdx.x * kConvWaves + wave) * (MT * 16);
    if (m0 >= M) return;   // the whole wave is past the volume (no barriers below)
    const int HW = a.H * a.W;
    int vz[MT], vy[MT], vx[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const size_t m = m0 + mt * 16 + row;
        if (m < M) {
            vz[mt] = (int)(m / HW);
            const int r = (int)(m - (size_t)vz[mt] * HW);
            vy[mt] = r / a.W;
            vx[mt] = r - vy[mt] * a.W;
        } else {
            vz[mt] = -4;   // every tap falls outside
            vy[mt] = 0;
            vx[mt] = 0;
        }
    }
    floatx4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    const int ca = a.src.ca, cin = a.src.ca + a.src.cb;
    const int Hh = a.H >> 1, Wh = a.W >> 1;
    const bf16x8 zero = as_bf16x8(u32x4{0u, 0u, 0u, 0u});
    for (int k0 = kg * 8; k0 < a.kpad; k0 += 32) {
        bf16x8 B[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) B[nt] = as_bf16x8(load16(a.wt + (size_t)(nt * 16 + row) * a.kpad + k0));
        bf16x8 A[MT];
        {
            const int t = k0 / cin, ci = k0 - t * cin;
            const int dz = t / 9 - 1, dy = (t / 3) % 3 - 1, dx = t % 3 - 1;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const int zz = vz[mt] + dz, yy = vy[mt] + dy, xx = vx[mt] + dx;
                A[mt] = zero;
                if (t < 27 && (unsigned)zz < (unsigned)a.D && (unsigned)yy < (unsigned)a.H &&
                    (unsigned)xx < (unsigned)a.W) {
                    const uint16_t* p;
                    if (ci < ca) {
                        const size_t v = a.src.a_half ? ((size_t)(zz >> 1) * Hh + (yy >> 1)) * Wh + (xx >> 1)
                                                      : ((size_t)zz * a.H + yy) * a.W + xx;
                        p = a.src.a + v * ca + ci;
                    } else {
                        p = a.src.b + (((size_t)zz * a.H + yy) * a.W + xx) * a.src.cb + (ci - ca);
                    }
                    A[mt] = as_bf16x8(load16(p));
                }
            }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[mt], B[nt], acc[mt][nt], 0, 0, 0);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int co = nt * 16 + row;
            const float b = a.bias ? a.bias[co] : 0.0f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const size_t m = m0 + mt * 16 + kg * 4 + r;
                if (m < M) {
                    float v = acc[mt][nt][r] + b;
                    if (a.relu) v = fmaxf(v, 0.0f);
                    a.out[m * a.cout + co] = f2bf(v);
                }
            }
        }
}

// ---- 3x3x3 convolution to 16 or 32 channels, LDS-staged bricks ----------
// A workgroup computes a kBZ x kBY x kBX brick of output voxels, all
// NT x 16 output channels.  Its input halo (kBZ + 2) x (kBY + 2) x (kBX + 2)
// is staged in LDS eight input channels at a time (one 16-byte cell per halo
// voxel), so that the 27 taps read each staged voxel from LDS instead of from
// memory.  An MFMA k step takes four taps of the chunk: lane group kg's A
// operand is its voxel's 8 channels at tap 4 s + kg, and its B operand the 8
// weights wt[co][tap * cin + ci ..] of the same tap, contiguous in the forward
// weight layout (the k order inside a step only has to agree between A and
// B).  The next chunk's weights and halo are loaded into registers while the
// current chunk's MFMAs run.  Wave w owns the brick's output rows
// (z = w, y = 0..7), two 16-voxel tiles each: the LDS reads of a step share one
// base address and differ by constant offsets.  The result goes through LDS
// (one 16-channel slice at a time) so that each voxel's channels leave in
// 16-byte stores.
constexpr int kBZ = kConvWaves, kBY = 8, kBX = 32;
constexpr int kHZ = kBZ + 2, kHY = kBY + 2, kHX = kBX + 2;
constexpr int kHaloCells = kHZ * kHY * kHX;                    // 2040
constexpr int kBrickVoxels = kBZ * kBY * kBX;                  // 1024
constexpr int kBrickTiles = kBrickVoxels / 16 / kConvWaves;    // 16 tiles of 16 voxels per wave
constexpr int kStage = (kHaloCells + kThreads - 1) / kThreads; // halo cells per thread
constexpr int kChunkSteps = (27 + 3) / 4;                      // k steps per 8-channel chunk
constexpr int kBrickLds = 2 * kBrickVoxels;                    // cells: >= the halo, = one output slice

template <int NT>
__global__ void __launch_bounds__(kThreads) conv3_brick_kernel(ConvArgs a, int nbx, int nby)
{
    static_assert(kBrickLds >= kHaloCells, "the output slice reuses the halo's LDS");
    __shared__ u32x4 lds[kBrickLds];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane & 15, kg = lane >> 4;
    const int bxi = blockIdx.x % nbx, rest = blockIdx.x / nbx;
    const int byi = rest % nby, bzi = rest / nby;
    const int x0 = bxi * kBX, y0 = byi * kBY, z0 = bzi * kBZ;
    const int ca = a.src.ca, cin = a.src.ca + a.src.cb;
    const int Hh = a.H >> 1, Wh = a.W >> 1;
    const u32x4 zero4 = u32x4{0u, 0u, 0u, 0u};

    floatx4 acc[kBrickTiles][NT];
#pragma unroll
    for (int t = 0; t < kBrickTiles; ++t)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[t][nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    // one chunk's weights (step st, tap 4 st + kg, output channel nt * 16 + row)
    // and halo cells, loaded into registers; the next chunk's loads are in
    // flight while the current chunk's MFMAs run
    u32x4 B[kChunkSteps][NT], cell[kStage];
    auto load_chunk = [&](int c0) {
#pragma unroll
        for (int st = 0; st < kChunkSteps; ++st) {
            const int tap = 4 * st + kg;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                B[st][nt] = tap < 27 ? load16(a.wt + (size_t)(nt * 16 + row) * a.kpad + tap * cin + c0) : zero4;
        }
#pragma unroll
        for (int k = 0; k < kStage; ++k) {
            const int e = k * kThreads + tid;
            cell[k] = zero4;
            if (e < kHaloCells) {
                const int hz = e / (kHY * kHX), r2 = e - hz * (kHY * kHX), hy = r2 / kHX, hx = r2 - hy * kHX;
                const int zz = z0 - 1 + hz, yy = y0 - 1 + hy, xx = x0 - 1 + hx;
                if ((unsigned)zz < (unsigned)a.D && (unsigned)yy < (unsigned)a.H && (unsigned)xx < (unsigned)a.W) {
                    const uint16_t* p;
                    if (c0 < ca) {
                        const size_t vi = a.src.a_half ? ((size_t)(zz >> 1) * Hh + (yy >> 1)) * Wh + (xx >> 1)
                                                       : ((size_t)zz * a.H + yy) * a.W + xx;
                        p = a.src.a + vi * ca + c0;
                    } else {
                        p = a.src.b + (((size_t)zz * a.H + yy) * a.W + xx) * a.src.cb + (c0 - ca);
                    }
                    cell[k] = load16(p);
                }
            }
        }
    };
    load_chunk(0);
    for (int c0 = 0; c0 < cin; c0 += 8) {
        __syncthreads();   // the previous chunk's reads of lds are done
#pragma unroll
        for (int k = 0; k < kStage; ++k) {
            const int e = k * kThreads + tid;
            if (e < kHaloCells) lds[e] = cell[k];
        }
        u32x4 Bc[kChunkSteps][NT];
#pragma unroll
        for (int st = 0; st < kChunkSteps; ++st)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) Bc[st][nt] = B[st][nt];
        __syncthreads();
        if (c0 + 8 < cin) load_chunk(c0 + 8);
#pragma unroll
        for (int st = 0; st < kChunkSteps; ++st) {
            const int tap = 4 * st + kg;
            const bool live = tap < 27;
            const int tc = live ? tap : 0;   // a valid address for the padding taps (B is zero there)
            const int dz = tc / 9, dy = (tc / 3) % 3, dx = tc % 3;
            const u32x4* base = lds + ((wave + dz) * kHY + dy) * kHX + dx + row;
#pragma unroll
            for (int t = 0; t < kBrickTiles; ++t) {
                u32x4 av = base[(t >> 1) * kHX + (t & 1) * 16];
                if (!live) av = zero4;
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    acc[t][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(av), as_bf16x8(Bc[st][nt]),
                                                                         acc[t][nt], 0, 0, 0);
            }
        }
    }
    // epilogue, one 16-channel slice at a time: bias, activation, bf16 into
    // LDS as [brick voxel][16 channels], then 16-byte stores of 8 channels
    uint16_t* slice = reinterpret_cast<uint16_t*>(lds);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int co = nt * 16 + row;
        const float b = a.bias ? a.bias[co] : 0.0f;
        __syncthreads();   // the last chunk's reads (or the previous slice's copy) are done
#pragma unroll
        for (int t = 0; t < kBrickTiles; ++t) {
            const int v0 = (wave * kBY + (t >> 1)) * kBX + (t & 1) * 16 + kg * 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = acc[t][nt][e] + b;
                if (a.relu) v = fmaxf(v, 0.0f);
                slice[(v0 + e) * 16 + row] = f2bf(v);
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kBrickLds / kThreads; ++k) {
            const int c = k * kThreads + tid;         // cell: voxel c / 2, channels 8 (c % 2) ..
            const int bv = c >> 1, bz = bv / (kBY * kBX), by = (bv / kBX) % kBY, bx = bv % kBX;
            const int z = z0 + bz, y = y0 + by, x = x0 + bx;
            if (z < a.D && y < a.H && x < a.W)
                *reinterpret_cast<u32x4*>(a.out + (((size_t)z * a.H + y) * a.W + x) * a.cout + nt * 16 + (c & 1) * 8) =
                    lds[c];
        }
    }
}

template <int NT, int MT>
void launch_conv(const ConvArgs& a, hipStream_t stream)
{
    const size_t M = (size_t)a.D * a.H * a.W;
    const size_t per_block = (size_t)kConvWaves * MT * 16;
    const dim3 grid((unsigned)((M + per_block - 1) / per_block));
    conv3_fwd_kernel<NT, MT><<<grid, kThreads, 0, stream>>>(a);
}

// ---- weight and bias gradient -------------------------------------------------
// A workgroup takes 16 input channels, all output channels (NT tiles of 16),
// all 27 taps and every chunk-th brick of kWZ x kWY x kWX voxels.  Both
// operands of the GEMM need 8 voxels of one channel per lane while memory
// holds 8 channels of one voxel: the input brick with its halo and the output
// gradient's brick are staged as they are ([voxel][16 channels], 16-byte
// cells) and read through ds_read_b64_tr_b16, which hands lane i of a 16-lane
// group column i of 4 voxels x 16 channels.  A tap is then a row and column
// offset into the halo, and the 27 taps read each staged voxel from LDS.  A
// 32-wide k step is one x row of the brick; lane group kg holds voxels
// 16 h + 4 kg + {0..3} (h = 0, 1) in both operands, so that one read of the
// wave covers 512 contiguous bytes (the k order only has to agree between A
// and B).  Wave w accumulates taps w, w + 4, ...; its slot past tap 26
// multiplies the gradient by one: the bias gradient.
// Bound by the LDS reads (two 8-byte reads a lane per MFMA and NT); the
// version that staged one tap's transposed operands through 2-byte LDS writes
// took 8.0 ms for the ten layers at 128^3, 27 passes over both operands.
constexpr int kWZ = 4, kWY = 4, kWX = 32;
constexpr int kWHZ = kWZ + 2, kWHY = kWY + 2, kWHX = kWX + 2;
constexpr int kWVoxels = kWZ * kWY * kWX;                       // 512
constexpr int kWHalo = kWHZ * kWHY * kWHX;                      // 1224
constexpr int kWTaps = (27 + kConvWaves - 1) / kConvWaves;      // tap slots per wave
constexpr int kMaxCout = 64;

struct WgradArgs {
    ConvSrc src;
    int D, H, W;
    const uint16_t* gy;
    int cout, cin16;
    int nbx, nby, bricks;
    float* partial;     // [chunk][27 * cout * cin16 weights, then cout biases]
};

typedef short i16x4 __attribute__((ext_vector_type(4)));
#ifdef __HIP_DEVICE_COMPILE__
#define ETN_LDS __attribute__((address_space(3)))
#else
#define ETN_LDS
#endif

// 8 voxels of one channel per lane (see above); cell: the lane's 8 bytes of
// the first 16 voxels, the second 16 are 512 bytes on
__device__ __forceinline__ bf16x8 load_voxels(const char* cell)
{
#ifdef __HIP_DEVICE_COMPILE__
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ETN_LDS i16x4*)(cell));
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ETN_LDS i16x4*)(cell + 512));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#else
    return as_bf16x8(*reinterpret_cast<const u32x4*>(cell));   // the host pass only parses this
#endif
}

template <int NT>
__global__ void __launch_bounds__(kThreads, NT == 4 ? 1 : 2) conv3_wgrad_kernel(WgradArgs w)
{
    __shared__ u32x4 xs[kWHalo * 2];          // [halo voxel][2 cells of 8 channels]
    __shared__ u32x4 gs[NT * kWVoxels * 2];   // [channel tile][voxel][2 cells]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 15, kg = lane >> 4;
    const int ci0 = blockIdx.y * 16;
    const int ca = w.src.ca, cin = w.src.ca + w.src.cb;
    const int Hh = w.H >> 1, Wh = w.W >> 1;
    const u32x4 zero4 = u32x4{0u, 0u, 0u, 0u};
    const bf16x8 ones = as_bf16x8(u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u});

    floatx4 acc[kWTaps][NT];
#pragma unroll
    for (int i = 0; i < kWTaps; ++i)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[i][nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    // the lane's cell of a row's first 16 voxels: voxel 4 kg + (lane & 15) / 4,
    // channels 4 (lane % 4) ..
    const int lane_cell = (4 * kg + (col >> 2)) * 32 + (col & 3) * 8;
    const char* xbase = reinterpret_cast<const char*>(xs) + lane_cell;
    const char* gbase = reinterpret_cast<const char*>(gs) + lane_cell;
    int tap_off[kWTaps];
#pragma unroll
    for (int i = 0; i < kWTaps; ++i) {
        const int t = wave + kConvWaves * i;
        tap_off[i] = (((t / 9) * kWHY + (t / 3) % 3) * kWHX + t % 3) * 32;
    }

    for (int b = blockIdx.x; b < w.bricks; b += gridDim.x) {
        const int bxi = b % w.nbx, rest = b / w.nbx, byi = rest % w.nby, bzi = rest / w.nby;
        const int x0 = bxi * kWX, y0 = byi * kWY, z0 = bzi * kWZ;
        __syncthreads();   // the previous brick's reads are done
        for (int e = tid; e < kWHalo * 2; e += kThreads) {
            const int v = e >> 1, c = ci0 + (e & 1) * 8;
            const int hz = v / (kWHY * kWHX), r2 = v - hz * (kWHY * kWHX), hy = r2 / kWHX, hx = r2 - hy * kWHX;
            const int zz = z0 - 1 + hz, yy = y0 - 1 + hy, xx = x0 - 1 + hx;
            u32x4 cell = zero4;
            if (c < cin && (unsigned)zz < (unsigned)w.D && (unsigned)yy < (unsigned)w.H && (unsigned)xx < (unsigned)w.W) {
                if (c < ca) {
                    const size_t vi = w.src.a_half ? ((size_t)(zz >> 1) * Hh + (yy >> 1)) * Wh + (xx >> 1)
                                                   : ((size_t)zz * w.H + yy) * w.W + xx;
                    cell = load16(w.src.a + vi * ca + c);
                } else {
                    cell = load16(w.src.b + (((size_t)zz * w.H + yy) * w.W + xx) * w.src.cb + (c - ca));
                }
            }
            xs[e] = cell;
        }
#pragma unroll
        for (int k = 0; k < NT * kWVoxels * 2 / kThreads; ++k) {
            const int e = k * kThreads + tid;
            const int v = e / (2 * NT), c = e - v * (2 * NT);
            const int z = z0 + v / (kWY * kWX), y = y0 + (v / kWX) % kWY, x = x0 + v % kWX;
            u32x4 cell = zero4;
            if (z < w.D && y < w.H && x < w.W) cell = load16(w.gy + (((size_t)z * w.H + y) * w.W + x) * w.cout + c * 8);
            gs[((c >> 1) * kWVoxels + v) * 2 + (c & 1)] = cell;
        }
        __syncthreads();
#pragma unroll 2
        for (int row = 0; row < kWZ * kWY; ++row) {
            bf16x8 A[NT];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) A[nt] = load_voxels(gbase + (nt * kWVoxels + row * kWX) * 32);
            const char* xrow = xbase + (((row / kWY) * kWHY + row % kWY) * kWHX) * 32;
#pragma unroll
            for (int i = 0; i < kWTaps; ++i) {
                const bool tap = i + 1 < kWTaps || wave + kConvWaves * i < 27;   // uniform in the wave
                const bf16x8 B = tap ? load_voxels(xrow + tap_off[i]) : ones;
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    acc[i][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[nt], B, acc[i][nt], 0, 0, 0);
            }
        }
    }
    float* out = w.partial + (size_t)blockIdx.x * ((size_t)27 * w.cout * w.cin16 + w.cout);
#pragma unroll
    for (int i = 0; i < kWTaps; ++i) {
        const int t = wave + kConvWaves * i;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int co = nt * 16 + kg * 4 + r;
                if (t < 27) out[((size_t)t * w.cout + co) * w.cin16 + ci0 + col] = acc[i][nt][r];
                else if (ci0 == 0 && col == 0) out[(size_t)27 * w.cout * w.cin16 + co] = acc[i][nt][r];
            }
    }
}

// Sum of `chunks` rows of n partial sums, rows `stride` apart: kSumLanes
// threads share a column, each adding every kSumLanes-th row in order, then
// the lanes are added in order (deterministic).  One thread per column left
// the few columns of a bias waiting on thousands of dependent loads: 3.0 ms
// of a 128^3 gradient, and 6.6 ms for the weights.
constexpr int kSumColumns = 32, kSumLanes = kThreads / kSumColumns;
template <typename Store>
__device__ __forceinline__ void sum_rows(const float* partial, int chunks, size_t stride, int n, Store&& store)
{
    __shared__ float red[kThreads];
    const int c = threadIdx.x % kSumColumns, l = threadIdx.x / kSumColumns;
    const int i = blockIdx.x * kSumColumns + c;
    float s = 0.0f;
    if (i < n) {
#pragma unroll 8
        for (int k = l; k < chunks; k += kSumLanes) s += partial[(size_t)k * stride + i];
    }
    red[threadIdx.x] = s;
    __syncthreads();
    if (l == 0 && i < n) {
        float t = 0.0f;
        for (int q = 0; q < kSumLanes; ++q) t += red[q * kSumColumns + c];
        store(i, t);
    }
}

__global__ void __launch_bounds__(kThreads) wgrad_reduce_kernel(const float* partial, int chunks, int cout, int cin,
                                                                int cin16, float* dw, float* db)
{
    const int nw = 27 * cout * cin16;
    sum_rows(partial, chunks, (size_t)nw + cout, nw + cout, [&](int i, float v) {
        if (i >= nw) {
            db[i - nw] = v;
            return;
        }
        const int t = i / (cout * cin16), r = i - t * cout * cin16, co = r / cin16, ci = r - co * cin16;
        if (ci < cin) dw[((size_t)co * 27 + t) * cin + ci] = v;
    });
}

__global__ void __launch_bounds__(kThreads) sum_partials_kernel(const float* partial, int chunks, int C, float* out)
{
    sum_rows(partial, chunks, (size_t)C, C, [&](int i, float v) { out[i] = v; });
}

__global__ void pack_weights_kernel(const float* w, int cout, int cin, int cin_pad, uint16_t* wt, int kpad,
                                    uint16_t* wb, int kpad_b)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cout * kpad) {
        const int co = i / kpad, k = i - co * kpad, t = k / cin_pad, ci = k - t * cin_pad;
        wt[i] = (t < 27 && ci < cin) ? f2bf(w[((size_t)co * 27 + t) * cin + ci]) : (uint16_t)0;
    }
    if (wb && i < cin * kpad_b) {
        const int ci = i / kpad_b, k = i - ci * kpad_b, t = k / cout, co = k - t * cout;
        wb[i] = t < 27 ? f2bf(w[((size_t)co * 27 + (26 - t)) * cin + ci]) : (uint16_t)0;
    }
}

__global__ void relu_backward_kernel(uint16_t* g, const uint16_t* y, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const uint16_t v = y[i];
        if ((v & 0x8000u) || (v & 0x7fffu) == 0) g[i] = 0;
    }
}

__global__ void pool2_kernel(const uint16_t* x, int D, int H, int W, int C, uint16_t* y)
{
    const int Dl = D / 2, Hl = H / 2, Wl = W / 2;
    const size_t n = (size_t)Dl * Hl * Wl * C;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int c = (int)(i % C);
        const size_t p = i / C;
        const int xl = (int)(p % Wl), yl = (int)((p / Wl) % Hl), zl = (int)(p / ((size_t)Wl * Hl));
        float s = 0.0f;
        for (int a = 0; a < 2; ++a)
            for (int b = 0; b < 2; ++b)
                for (int e = 0; e < 2; ++e)
                    s += bf2f(x[((((size_t)(2 * zl + a) * H) + 2 * yl + b) * W + 2 * xl + e) * C + c]);
        y[i] = f2bf(s * 0.125f);
    }
}

__global__ void pool2_backward_kernel(const uint16_t* gl, int D, int H, int W, int C, uint16_t* g, int accumulate)
{
    const size_t n = (size_t)D * H * W * C;
    const int Hl = H / 2, Wl = W / 2;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int c = (int)(i % C);
        const size_t m = i / C;
        const int x = (int)(m % W), y = (int)((m / W) % H), z = (int)(m / ((size_t)W * H));
        const float v = bf2f(gl[(((size_t)(z / 2) * Hl + y / 2) * Wl + x / 2) * C + c]) * 0.125f;
        g[i] = f2bf(accumulate ? bf2f(g[i]) + v : v);
    }
}

__global__ void up2_backward_kernel(const uint16_t* g, int stride, int c0, int D, int H, int W, int C, uint16_t* gl)
{
    const int Dl = D / 2, Hl = H / 2, Wl = W / 2;
    const size_t n = (size_t)Dl * Hl * Wl * C;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int c = (int)(i % C);
        const size_t p = i / C;
        const int xl = (int)(p % Wl), yl = (int)((p / Wl) % Hl), zl = (int)(p / ((size_t)Wl * Hl));
        float s = 0.0f;
        for (int a = 0; a < 2; ++a)
            for (int b = 0; b < 2; ++b)
                for (int e = 0; e < 2; ++e)
                    s += bf2f(g[((((size_t)(2 * zl + a) * H) + 2 * yl + b) * W + 2 * xl + e) * stride + c0 + c]);
        gl[i] = f2bf(s);
    }
}

__global__ void take_channels_kernel(const uint16_t* g, int stride, int c0, size_t voxels, int C, uint16_t* dst,
                                     int accumulate)
{
    const size_t n = voxels * C;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const size_t m = i / C;
        const int c = (int)(i - m * C);
        const float v = bf2f(g[m * stride + c0 + c]);
        dst[i] = f2bf(accumulate ? bf2f(dst[i]) + v : v);
    }
}

__global__ void pack_input_kernel(const float* x, float scale, const float* d, float dscale, size_t n, uint16_t* y)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const uint32_t a = f2bf(x[i] * scale), b = d ? f2bf(d[i] * dscale) : 0u;
        *reinterpret_cast<u32x4*>(y + 8 * i) = u32x4{a | (b << 16), 0u, 0u, 0u};
    }
}

__global__ void head_forward_kernel(const uint16_t* d1, const float* x, float scale, const float* hw, const float* hb,
                                    size_t n, float* pred)
{
    for (size_t m = (size_t)blockIdx.x * blockDim.x + threadIdx.x; m < n; m += (size_t)gridDim.x * blockDim.x) {
        const u32x4 a = load16(d1 + m * 16), b = load16(d1 + m * 16 + 8);
        float s = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s += hw[2 * e] * bf2f((uint16_t)(a[e] & 0xffffu)) + hw[2 * e + 1] * bf2f((uint16_t)(a[e] >> 16));
            s += hw[8 + 2 * e] * bf2f((uint16_t)(b[e] & 0xffffu)) + hw[9 + 2 * e] * bf2f((uint16_t)(b[e] >> 16));
        }
        pred[m] = x[m] * scale + (s + hb[0]);
    }
}

__global__ void unscale_kernel(const float* pred, const float* x, float scale, size_t n, float* out)
{
    for (size_t m = (size_t)blockIdx.x * blockDim.x + threadIdx.x; m < n; m += (size_t)gridDim.x * blockDim.x)
        out[m] = x[m] + (pred[m] - x[m] * scale) / scale;
}

constexpr int kRedBlocks = 1024;

__global__ void mse_partial_kernel(const float* pred, const float* target, float scale, size_t n, float* g,
                                   double* partial)
{
    __shared__ double red[kThreads];
    double s = 0.0;
    const float inv = 2.0f / (float)n;
    for (size_t m = (size_t)blockIdx.x * blockDim.x + threadIdx.x; m < n; m += (size_t)gridDim.x * blockDim.x) {
        const float r = pred[m] - target[m] * scale;
        g[m] = r * inv;
        s += (double)r * (double)r;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = kThreads / 2; w > 0; w /= 2) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void __launch_bounds__(kThreads) mse_final_kernel(const double* partial, int blocks, size_t n, double* loss)
{
    __shared__ double red[kThreads];
    double s = 0.0;
    for (int b = threadIdx.x; b < blocks; b += kThreads) s += partial[b];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = kThreads / 2; w > 0; w /= 2) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *loss = red[0] / (double)n;
}

__global__ void head_backward_kernel(const uint16_t* d1, const float* gp, const float* hw, size_t n, uint16_t* gd1,
                                     float* partial)
{
    __shared__ float red[kThreads * 17];
    float s[17];
#pragma unroll
    for (int c = 0; c < 17; ++c) s[c] = 0.0f;
    for (size_t m = (size_t)blockIdx.x * blockDim.x + threadIdx.x; m < n; m += (size_t)gridDim.x * blockDim.x) {
        const float g = gp[m];
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            s[c] += g * bf2f(d1[m * 16 + c]);
            gd1[m * 16 + c] = f2bf(g * hw[c]);
        }
        s[16] += g;
    }
#pragma unroll
    for (int c = 0; c < 17; ++c) red[c * kThreads + threadIdx.x] = s[c];
    __syncthreads();
    if (threadIdx.x < 17) {
        float t = 0.0f;
        for (int q = 0; q < kThreads; ++q) t += red[threadIdx.x * kThreads + q];
        partial[(size_t)blockIdx.x * 17 + threadIdx.x] = t;
    }
}

__global__ void adam_kernel(float* p, const float* g, float* m, float* v, size_t n, float lr, float b1, float b2,
                            float eps, float bc1, float bc2)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.0f - b1) * gi;
        const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        p[i] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
    }
}

unsigned grid_for(size_t n)
{
    return (unsigned)std::max<size_t>(1, std::min<size_t>((n + kThreads - 1) / kThreads, 65536));
}

}  // namespace

void conv3_forward(const ConvArgs& a, hipStream_t stream)
{
    if (a.src.ca < 8 || (a.src.ca % 8) || (a.src.cb % 8)) fail("conv3: input channels must be multiples of 8");
    if (a.kpad != kpad_for(a.src.ca + a.src.cb)) fail("conv3: weight row length mismatch");
    if (a.src.a_half && ((a.D | a.H | a.W) & 1)) fail("conv3: upsampled input needs even sizes");
    const int nbx = (a.W + kBX - 1) / kBX, nby = (a.H + kBY - 1) / kBY, nbz = (a.D + kBZ - 1) / kBZ;
    const unsigned bricks = (unsigned)(nbx * nby * nbz);
    switch (a.cout) {
        case 16: conv3_brick_kernel<1><<<bricks, kThreads, 0, stream>>>(a, nbx, nby); break;
        case 32: conv3_brick_kernel<2><<<bricks, kThreads, 0, stream>>>(a, nbx, nby); break;
        case 48: launch_conv<3, 2>(a, stream); break;
        case 64: launch_conv<4, 2>(a, stream); break;
        case 96: launch_conv<6, 2>(a, stream); break;
        default: fail("conv3: output channels must be 16, 32, 48, 64 or 96");
    }
    hip_check(hipGetLastError(), "conv3 forward launch");
}

int wgrad_chunks(int D, int H, int W, int cin)
{
    // two workgroups per CU over all channel chunks, at most one per brick:
    // more only adds partial sums to write and read back
    const int bricks = ((W + kWX - 1) / kWX) * ((H + kWY - 1) / kWY) * ((D + kWZ - 1) / kWZ);
    return std::min(bricks, std::max(1, 512 / ((cin + 15) / 16)));
}

size_t wgrad_partial_floats(int D, int H, int W, int cin, int cout)
{
    return (size_t)wgrad_chunks(D, H, W, cin) * ((size_t)27 * cout * ((cin + 15) / 16 * 16) + cout);
}

void conv3_weight_grad(const ConvSrc& src, int D, int H, int W, const uint16_t* gy, int cin, int cout, float* partial,
                       float* dw, float* db, hipStream_t stream)
{
    if (cout % 16 || cout > kMaxCout || cout == 48 || src.ca % 8 || src.cb % 8 || cin > src.ca + src.cb)
        fail("conv3 weight gradient: channel counts");
    const int cin16 = (src.ca + src.cb + 15) / 16 * 16, chunks = wgrad_chunks(D, H, W, src.ca + src.cb);
    const int nbx = (W + kWX - 1) / kWX, nby = (H + kWY - 1) / kWY, nbz = (D + kWZ - 1) / kWZ;
    WgradArgs w{src, D, H, W, gy, cout, cin16, nbx, nby, nbx * nby * nbz, partial};
    const dim3 grid((unsigned)chunks, (unsigned)(cin16 / 16));
    switch (cout / 16) {
        case 1: conv3_wgrad_kernel<1><<<grid, kThreads, 0, stream>>>(w); break;
        case 2: conv3_wgrad_kernel<2><<<grid, kThreads, 0, stream>>>(w); break;
        default: conv3_wgrad_kernel<4><<<grid, kThreads, 0, stream>>>(w); break;
    }
    const int n = 27 * cout * cin16 + cout;
    wgrad_reduce_kernel<<<(n + kSumColumns - 1) / kSumColumns, kThreads, 0, stream>>>(partial, chunks, cout, cin, cin16,
                                                                                     dw, db);
    hip_check(hipGetLastError(), "conv3 weight gradient launch");
}

void pack_weights(const float* w, int cout, int cin, int cin_pad, uint16_t* wt, uint16_t* wb, hipStream_t stream)
{
    const int kpad = kpad_for(cin_pad), kpad_b = kpad_for(cout);
    const int n = std::max(cout * kpad, wb ? cin * kpad_b : 0);
    pack_weights_kernel<<<(n + kThreads - 1) / kThreads, kThreads, 0, stream>>>(w, cout, cin, cin_pad, wt, kpad, wb,
                                                                               kpad_b);
    hip_check(hipGetLastError(), "weight packing launch");
}

void relu_backward(uint16_t* g, const uint16_t* y, size_t count, hipStream_t stream)
{
    relu_backward_kernel<<<grid_for(count), kThreads, 0, stream>>>(g, y, count);
}

void pool2(const uint16_t* x, int D, int H, int W, int C, uint16_t* y, hipStream_t stream)
{
    pool2_kernel<<<grid_for((size_t)D * H * W * C / 8), kThreads, 0, stream>>>(x, D, H, W, C, y);
}

void pool2_backward(const uint16_t* g_low, int D, int H, int W, int C, uint16_t* g_full, int accumulate,
                    hipStream_t stream)
{
    pool2_backward_kernel<<<grid_for((size_t)D * H * W * C), kThreads, 0, stream>>>(g_low, D, H, W, C, g_full,
                                                                                    accumulate);
}

void up2_backward(const uint16_t* g, int stride, int c0, int D, int H, int W, int C, uint16_t* g_low,
                  hipStream_t stream)
{
    up2_backward_kernel<<<grid_for((size_t)D * H * W * C / 8), kThreads, 0, stream>>>(g, stride, c0, D, H, W, C,
                                                                                      g_low);
}

void take_channels(const uint16_t* g, int stride, int c0, size_t voxels, int C, uint16_t* dst, int accumulate,
                   hipStream_t stream)
{
    take_channels_kernel<<<grid_for(voxels * C), kThreads, 0, stream>>>(g, stride, c0, voxels, C, dst, accumulate);
}

void pack_input(const float* x, float scale, const float* d, float dscale, size_t count, uint16_t* y,
                hipStream_t stream)
{
    pack_input_kernel<<<grid_for(count), kThreads, 0, stream>>>(x, scale, d, dscale, count, y);
}

void head_forward(const uint16_t* d1, const float* x, float scale, const float* hw, const float* hb, size_t voxels,
                  float* pred, hipStream_t stream)
{
    head_forward_kernel<<<grid_for(voxels), kThreads, 0, stream>>>(d1, x, scale, hw, hb, voxels, pred);
}

void unscale_prediction(const float* pred, const float* x, float scale, size_t voxels, float* out, hipStream_t stream)
{
    unscale_kernel<<<grid_for(voxels), kThreads, 0, stream>>>(pred, x, scale, voxels, out);
}

void mse_loss(const float* pred, const float* target, float scale, size_t voxels, float* g_pred, double* partial,
              double* loss, hipStream_t stream)
{
    mse_partial_kernel<<<kRedBlocks, kThreads, 0, stream>>>(pred, target, scale, voxels, g_pred, partial);
    mse_final_kernel<<<1, kThreads, 0, stream>>>(partial, kRedBlocks, voxels, loss);
}

void head_backward(const uint16_t* d1, const float* g_pred, const float* hw, size_t voxels, uint16_t* g_d1,
                   float* partial, float* ghw_ghb, hipStream_t stream)
{
    head_backward_kernel<<<kRedBlocks, kThreads, 0, stream>>>(d1, g_pred, hw, voxels, g_d1, partial);
    sum_partials_kernel<<<1, kThreads, 0, stream>>>(partial, kRedBlocks, 17, ghw_ghb);
}

void adam_step(float* p, const float* g, float* m, float* v, size_t count, float lr, float beta1, float beta2,
               float eps, float bc1, float bc2, hipStream_t stream)
{
    adam_kernel<<<grid_for(count), kThreads, 0, stream>>>(p, g, m, v, count, lr, beta1, beta2, eps, bc1, bc2);
}

}  // namespace nn
}  // namespace etn
