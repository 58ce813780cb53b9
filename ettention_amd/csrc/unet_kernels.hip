// Learned correction network kernels (see unet_kernels.hpp).
//
// The 3x3x3 convolutions are implicit GEMMs on the matrix cores
// (v_mfma_f32_16x16x32_bf16, FP32 accumulation): output channels are the rows,
// voxels the columns, taps x input channels the reduction.  Lane layouts
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

__device__ __forceinline__ uint16_t f2bf(float f) { return dev::BF16::pack(f); }

__device__ __forceinline__ u32x4 load16(const uint16_t* p) { return *reinterpret_cast<const u32x4*>(p); }
__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

constexpr int kConvWaves = 4;
constexpr int kThreads = 256;

// 1 where a stored activation is positive: the derivative of the ReLU behind it
__device__ __forceinline__ bool positive(uint16_t h) { return !(h & 0x8000u) && (h & 0x7fffu) != 0; }
// a pair of bf16 values with the ones whose activation is not positive set to zero
__device__ __forceinline__ uint32_t gated(uint32_t pair, uint32_t act)
{
    return (positive((uint16_t)(act & 0xffffu)) ? pair & 0xffffu : 0u) |
           (positive((uint16_t)(act >> 16)) ? pair & 0xffff0000u : 0u);
}

// ---- 3x3x3 convolution on LDS-staged bricks -------------------------------
// A workgroup computes a kBZ x kBY x kBX brick of output voxels and NC x 16
// output channels (blockIdx.y: which); each of its 8 NC waves owns 4 z x 2 y
// rows of 16 voxels and 16 channels, whose sums stay in registers.  The input
// brick with its halo is staged in LDS 16 channels at a time as two arrays of
// 16-byte cells (channels 0-7 and 8-15), with the chunk's weights behind it.
// The weights are the GEMM's rows and the voxels its columns, so that a lane
// ends with 4 consecutive channels of one voxel and stores 8 bytes without a
// pass through LDS.
// A 32-wide k step holds two taps of 16 channels (lane group kg: tap kg / 2,
// channels 8 (kg % 2) ..), chosen so that a voxel operand depends only on the
// input row it starts at and serves every output row whose taps it holds:
//   F1(r): taps dx = 0 and 1 of input row r,     used with dy = 0, 1, 2;
//   F2(r): tap dx = 2 of input rows r and r + 1, used with dy = 0 and 1 (P)
//          and with dy = 1 and 2 (Q).
// The weight of dx = 2, dy = 1, which both hold, is halved in each (exact: a power
// of two; a zero in one of them would turn an infinite voxel into NaN, and the ReLU
// that into 0).
// That is 5 steps per dz and output row (15 for the 27 taps, 0.9 of the
// products wanted) and 7 LDS reads for 10 MFMAs; a step of four arbitrary taps
// of 8 channels took one read per MFMA.  What bounds it besides the MFMAs is
// everything around them: a wave has 120 MFMAs a chunk (1920 cycles), so the
// halo's addresses are scalars (a wave stages whole rows; per-cell indices cost
// more VALU time than the MFMAs take), and 128 VGPRs keep four waves a SIMD,
// two workgroups a CU, for one to load while the other computes.  Measured at
// 256^3 (prediction 4.08 -> 2.27 ms): 48 to 16 channels 1.13 -> 0.80 ms (875
// TFLOP/s of its 27 taps), 16 to 16 with the pooling in the epilogue 0.35 ms
// (1.2 GB, 3.4 TB/s).
constexpr int kBZ = 4, kBY = 8, kBX = 32;
constexpr int kHZ = kBZ + 2, kHY = kBY + 2, kHX = kBX + 2;
constexpr int kHaloRows = kHZ * kHY;          // 60
constexpr int kHaloCells = kHaloRows * kHX;   // 2040
// Cells between the two channel halves.  A multiple of 16: lane groups 0 and 1
// (2 and 3) of a read are served together, and with the same position modulo
// the 256 bytes of the banks they do not collide (4.1 cycles a read of the
// wave, 8.0 with any other distance, 2040 among them).
constexpr int kPlane = (kHaloCells + 15) / 16 * 16;
constexpr int kConvThreads = 512;
constexpr int kXcds = 8;

// What a convolution does with its sums (besides bias and activation).
enum Epilogue {
    kStore,      // out, optionally gated
    kPool,       // out, and its 2 x 2 x 2 averages
    kChildren,   // the sums over 2 x 2 x 2 voxels, gated, instead of out
    kHead        // the 1 x 1 x 1 head's prediction; out only where it is wanted
};

// Brick of workgroup b of `groups` (a multiple of kXcds): the bricks of an XCD
// are consecutive (workgroup b runs on XCD b mod 8), so that neighbours read
// their shared halo from one L2.
__device__ __forceinline__ int brick_of(int b, int groups) { return b % kXcds * (groups / kXcds) + b / kXcds; }

template <int NC, Epilogue kEpi>
__global__ void __launch_bounds__(kConvThreads * NC, 4) conv3_brick_kernel(ConvArgs a, int nbx, int nby, int bricks)
{
    constexpr int kT = kConvThreads * NC, kWaves = kT / 64;
    __shared__ u32x4 lds[2 * kPlane];
    __shared__ u32x4 wlds[NC * kConvFrags * 64];   // the chunk's weights
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, kg = lane >> 4;
    const int brick = brick_of(blockIdx.x, gridDim.x);
    if (brick >= bricks) return;
    const int bxi = brick % nbx, rest = brick / nbx, byi = rest % nby, bzi = rest / nby;
    const int x0 = bxi * kBX, y0 = byi * kBY, z0 = bzi * kBZ;
    const int wx = (wave & 1) * 16, wy = (wave >> 1 & 3) * 2;   // the wave's voxels and rows in the brick
    const int ca = a.src.ca, cin = a.src.ca + a.src.cb;
    const int Hh = a.H >> 1, Wh = a.W >> 1;
    const u32x4 zero4 = u32x4{0u, 0u, 0u, 0u};
    const int tiles = a.cout / 16, tile = blockIdx.y * NC + (wave >> 3);

    // the lane's first channel and its bias (the sums start there)
    const int c = tile * 16 + kg * 4;
    floatx4 acc[kBZ][2];
    {
        floatx4 bias = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        if (a.bias) {
#pragma unroll
            for (int r = 0; r < 4; ++r) bias[r] = a.bias[c + r];
        }
#pragma unroll
        for (int z = 0; z < kBZ; ++z) acc[z][0] = acc[z][1] = bias;
    }

    // A wave stages halo rows wave, wave + kWaves, ...: lanes take the cells of
    // voxels 0 .. 31 (voxel lane / 2, channel half lane % 2), whose addresses are
    // the row's scalar one and the lane's offset; threads 0 .. 239 take voxels
    // 32 and 33 of the 60 rows.  Cells outside the volume read a valid address
    // and are zeroed on their way to LDS: a branch or a select at the load would
    // wait for it on the spot.
    constexpr int kRows = (kHaloRows + kWaves - 1) / kWaves;
    constexpr int kWStage = (NC * kConvFrags * 64 + kT - 1) / kT;
    u32x4 cell[kRows], edge, wcell[kWStage];
    const int hx = x0 - 1 + (lane >> 1), erow = tid >> 2, ehx = x0 + 31 + (tid >> 1 & 1);
    const int ehy = y0 - 1 + erow % kHY, ehz = z0 - 1 + erow / kHY;
    const bool hx_in = (unsigned)hx < (unsigned)a.W;
    const bool edge_in = erow < kHaloRows && ehx < a.W && (unsigned)ehy < (unsigned)a.H && (unsigned)ehz < (unsigned)a.D;
    auto row_y = [&](int k) { return y0 - 1 + (wave + k * kWaves) % kHY; };
    auto row_z = [&](int k) { return z0 - 1 + (wave + k * kWaves) / kHY; };
    auto load_chunk = [&](int c0) {
        const bool from_a = c0 < ca;
        const int cs = (from_a ? ca : a.src.cb) / 8;   // cells per voxel
        const u32x4* src = reinterpret_cast<const u32x4*>(from_a ? a.src.a + c0 : a.src.b + (c0 - ca));
        const int shift = from_a && a.src.a_half ? 1 : 0;
        const int Hs = shift ? Hh : a.H, Ws = shift ? Wh : a.W;
        const uint32_t at = (uint32_t)((hx_in ? hx >> shift : 0) * cs + (lane & 1));
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            const int y = min(max(row_y(k), 0), a.H - 1) >> shift, z = min(max(row_z(k), 0), a.D - 1) >> shift;
            cell[k] = (src + ((size_t)z * Hs + y) * Ws * cs)[at];
        }
        const size_t ev = edge_in ? ((size_t)(ehz >> shift) * Hs + (ehy >> shift)) * Ws + (ehx >> shift) : 0;
        edge = src[ev * cs + (tid & 1)];
        const u32x4* w = reinterpret_cast<const u32x4*>(a.wt) +
                         ((size_t)(c0 / 16) * tiles + blockIdx.y * NC) * (kConvFrags * 64);
#pragma unroll
        for (int k = 0; k < kWStage; ++k) wcell[k] = w[min(k * kT + tid, NC * kConvFrags * 64 - 1)];
    };
    load_chunk(0);
    // the lane's cell of F1(row 0) and F2(row 0) in halo slice 0, its weights
    const u32x4* half = lds + (kg & 1) * kPlane + wy * kHX + wx + col;
    const u32x4* f1 = half + (kg >> 1);
    const u32x4* f2 = half + (kg >> 1) * kHX + 2;
    const u32x4* wf = wlds + (wave >> 3) * (kConvFrags * 64) + lane;
    for (int c0 = 0; c0 < cin; c0 += 16) {
        __syncthreads();   // the previous chunk's reads are done
        u32x4* to = lds + (lane & 1) * kPlane + (lane >> 1) + wave * kHX;
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            const bool in = (unsigned)row_y(k) < (unsigned)a.H && (unsigned)row_z(k) < (unsigned)a.D && hx_in;
            if (wave + k * kWaves < kHaloRows) to[k * kWaves * kHX] = in ? cell[k] : zero4;
        }
        if (erow < kHaloRows) lds[(tid & 1) * kPlane + erow * kHX + 32 + (tid >> 1 & 1)] = edge_in ? edge : zero4;
#pragma unroll
        for (int k = 0; k < kWStage; ++k) {
            const int e = k * kT + tid;
            if (e < NC * kConvFrags * 64) wlds[e] = wcell[k];
        }
        __syncthreads();
        if (c0 + 16 < cin) load_chunk(c0 + 16);
#pragma unroll 1
        for (int dz = 0; dz < 3; ++dz) {
            bf16x8 w[kConvFrags / 3];
#pragma unroll
            for (int f = 0; f < kConvFrags / 3; ++f) w[f] = as_bf16x8(wf[(dz * (kConvFrags / 3) + f) * 64]);
#pragma unroll
            for (int z = 0; z < kBZ; ++z) {
                const u32x4* r1 = f1 + (z + dz) * (kHY * kHX);
                const u32x4* r2 = f2 + (z + dz) * (kHY * kHX);
                bf16x8 F1[4], F2[3];
#pragma unroll
                for (int r = 0; r < 4; ++r) F1[r] = as_bf16x8(r1[r * kHX]);
#pragma unroll
                for (int r = 0; r < 3; ++r) F2[r] = as_bf16x8(r2[r * kHX]);
#pragma unroll
                for (int f = 0; f < kConvFrags / 3; ++f)
#pragma unroll
                    for (int y = 0; y < 2; ++y)
                        acc[z][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[f], f < 3 ? F1[y + f] : F2[y + f - 3],
                                                                            acc[z][y], 0, 0, 0);
            }
        }
    }

    // rows are uniform in the wave: a row's address is a scalar plus the lane's
    // offset
    const int x = x0 + wx + col;
    const bool xin = x < a.W;
    const uint32_t at = (uint32_t)(x * a.cout + c), at_low = (uint32_t)((x >> 1) * a.cout + c);
    auto row = [&](int z, int y) { return ((size_t)(z0 + z) * a.H + (y0 + wy + y)) * a.W; };
    auto row_low = [&](int z) { return ((size_t)((z0 + z) >> 1) * Hh + ((y0 + wy) >> 1)) * Wh; };
    auto row_in = [&](int z, int y) { return z0 + z < a.D && y0 + wy + y < a.H; };
    // the gates of all the lane's voxels, in flight together
    [[maybe_unused]] uint2 gate[kEpi == kStore ? kBZ * 2 : kEpi == kChildren ? kBZ / 2 : 1];
    if constexpr (kEpi == kStore) {
        if (a.gate && xin) {
#pragma unroll
            for (int i = 0; i < kBZ * 2; ++i)
                if (row_in(i / 2, i % 2))
                    gate[i] = *reinterpret_cast<const uint2*>(a.gate + row(i / 2, i % 2) * a.cout + at);
        }
    }
    if constexpr (kEpi == kChildren) {
        if (a.gate && xin) {
#pragma unroll
            for (int i = 0; i < kBZ / 2; ++i)
                if (row_in(2 * i, 0)) gate[i] = *reinterpret_cast<const uint2*>(a.gate + row_low(2 * i) * a.cout + at_low);
        }
    }
#pragma unroll
    for (int z = 0; z < kBZ; ++z)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            floatx4& v = acc[z][y];
            if (a.relu) {
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = fmaxf(v[r], 0.0f);
            }
            if constexpr (kEpi == kChildren) continue;
            uint2 p = make_uint2(dev::BF16::pack2(v[0], v[1]), dev::BF16::pack2(v[2], v[3]));
            if constexpr (kEpi == kStore) {
                if (a.gate) p = make_uint2(gated(p.x, gate[z * 2 + y].x), gated(p.y, gate[z * 2 + y].y));
            }
            if (row_in(z, y) && xin && (kEpi != kHead || a.out))
                *reinterpret_cast<uint2*>(a.out + row(z, y) * a.cout + at) = p;
            if constexpr (kEpi == kPool || kEpi == kHead) {
                // what follows reads the stored (rounded) values
                float t[4];
                dev::BF16::unpack2(p.x, t[0], t[1]);
                dev::BF16::unpack2(p.y, t[2], t[3]);
                v = floatx4{t[0], t[1], t[2], t[3]};
            }
        }
    if constexpr (kEpi == kHead) {
        const bool mine = xin && kg == 0;
        float xv[kBZ * 2];
#pragma unroll
        for (int i = 0; i < kBZ * 2; ++i)
            if (mine && row_in(i / 2, i % 2)) xv[i] = (a.x + row(i / 2, i % 2))[(uint32_t)x];
#pragma unroll
        for (int i = 0; i < kBZ * 2; ++i) {
            const floatx4 v = acc[i / 2][i % 2];
            float s = a.head[c] * v[0];
#pragma unroll
            for (int r = 1; r < 4; ++r) s = fmaf(a.head[c + r], v[r], s);
            s += __shfl_xor(s, 16);
            s += __shfl_xor(s, 32);
            if (mine && row_in(i / 2, i % 2)) {
                const float xs = xv[i] * a.scale;
                const float pred = xs + (s + a.head[16]);
                (a.pred + row(i / 2, i % 2))[(uint32_t)x] = a.unscale ? xv[i] + (pred - xs) / a.scale : pred;
            }
        }
    }
    if constexpr (kEpi == kPool || kEpi == kChildren) {
        uint16_t* low = kEpi == kPool ? a.pool : a.out;
#pragma unroll
        for (int z = 0; z < kBZ; z += 2) {
            floatx4 s = (acc[z][0] + acc[z][1]) + (acc[z + 1][0] + acc[z + 1][1]);
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] += __shfl_xor(s[r], 1);
            if (kEpi == kPool) s *= 0.125f;
            if (row_in(z, 0) && xin && (col & 1) == 0) {   // (z, y and the sizes are even)
                uint2 p = make_uint2(dev::BF16::pack2(s[0], s[1]), dev::BF16::pack2(s[2], s[3]));
                if constexpr (kEpi == kChildren) {
                    if (a.gate) p = make_uint2(gated(p.x, gate[z / 2].x), gated(p.y, gate[z / 2].y));
                }
                *reinterpret_cast<uint2*>(low + row_low(z) * a.cout + at_low) = p;
            }
        }
    }
}

// ---- first layer: (x, d) to 16 channels -----------------------------------
// Reads the fp32 volumes themselves and keeps the halo in LDS as one 4-byte
// bf16 pair per voxel.  A lane's 8 operands are 4 consecutive voxels of one
// input row, the fourth and the rows past the ninth zero: 3 k steps for the 27
// taps of 2 channels, where the two channels padded to 8 took 7 and a 16-byte
// cell per voxel written and read back first (pack_input).  Bound by its
// 32-byte output per voxel: 0.20 ms at 256^3, 3.4 TB/s.
__global__ void __launch_bounds__(kThreads, 4) conv3_first_kernel(const float* __restrict__ xv, float scale,
                                                                  const float* __restrict__ dv, float dscale, int D,
                                                                  int H, int W, const uint16_t* __restrict__ wt,
                                                                  const float* __restrict__ bias, uint16_t* out, int nbx,
                                                                  int nby, int bricks)
{
    __shared__ uint32_t lds[kHaloCells];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 15, kg = lane >> 4;
    const int brick = brick_of(blockIdx.x, gridDim.x);
    if (brick >= bricks) return;
    const int bxi = brick % nbx, rest = brick / nbx, byi = rest % nby, bzi = rest / nby;
    const int x0 = bxi * kBX, y0 = byi * kBY, z0 = bzi * kBZ;
    const int wy = (wave >> 1) * 4, wx = (wave & 1) * 16;
#pragma unroll
    for (int k = 0; k < (kHaloCells + kThreads - 1) / kThreads; ++k) {
        const int v = k * kThreads + tid;
        const int hz = v / (kHY * kHX), r2 = v - hz * (kHY * kHX), hy = r2 / kHX, hx = r2 - hy * kHX;
        const int zz = z0 - 1 + hz, yy = y0 - 1 + hy, xx = x0 - 1 + hx;
        uint32_t pair = 0u;
        if ((unsigned)zz < (unsigned)D && (unsigned)yy < (unsigned)H && (unsigned)xx < (unsigned)W) {
            const size_t m = ((size_t)zz * H + yy) * W + xx;
            pair = dev::BF16::pack2(xv[m] * scale, dv ? dv[m] * dscale : 0.0f);
        }
        if (v < kHaloCells) lds[v] = pair;
    }
    bf16x8 w[3];
#pragma unroll
    for (int s = 0; s < 3; ++s) w[s] = as_bf16x8(load16(wt + (s * 64 + lane) * 8));
    float b[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) b[r] = bias[kg * 4 + r];
    __syncthreads();
    // step s, lane group kg: input row (dz, dy) = row 4 s + kg of the 3 x 3
    int row_off[3];
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        const int g = min(4 * s + kg, 8);
        row_off[s] = ((g / 3) * kHY + g % 3) * kHX;
    }
    const int x = x0 + wx + col;
#pragma unroll
    for (int z = 0; z < kBZ; ++z)
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            const uint32_t* at = lds + (z * kHY + wy + y) * kHX + wx + col;
            floatx4 acc = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < 3; ++s) {
                const uint32_t* p = at + row_off[s];
                u32x4 f = u32x4{p[0], p[1], p[2], 0u};
                if (4 * s + kg > 8) f = u32x4{0u, 0u, 0u, 0u};
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s], as_bf16x8(f), acc, 0, 0, 0);
            }
            const int zz = z0 + z, yy = y0 + wy + y;
            if (zz < D && yy < H && x < W) {
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = fmaxf(acc[r] + b[r], 0.0f);
                *reinterpret_cast<uint2*>(out + (((size_t)zz * H + yy) * W + x) * 16 + kg * 4) =
                    make_uint2(dev::BF16::pack2(v[0], v[1]), dev::BF16::pack2(v[2], v[3]));
            }
        }
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

    // the thread's share of a brick, loaded into registers while the brick
    // before it is worked on (cells outside the volume: a valid address, zeroed
    // on their way to LDS)
    const bool from_a = ci0 < ca;
    const int cs = from_a ? ca : w.src.cb;
    const uint16_t* src = from_a ? w.src.a + ci0 : w.src.b + (ci0 - ca);
    const int shift = from_a && w.src.a_half ? 1 : 0;
    const int Hs = shift ? Hh : w.H, Ws = shift ? Wh : w.W;
    constexpr int kWStage = (kWHalo * 2 + kThreads - 1) / kThreads, kGStage = NT * kWVoxels * 2 / kThreads;
    u32x4 xcell[kWStage], gcell[kGStage];
    uint32_t xin = 0u, gin = 0u;   // bit k: cell k lies in the volume
    auto load_brick = [&](int b) {
        xin = gin = 0u;
        const int bxi = b % w.nbx, rest = b / w.nbx, byi = rest % w.nby, bzi = rest / w.nby;
        const int x0 = bxi * kWX, y0 = byi * kWY, z0 = bzi * kWZ;
#pragma unroll
        for (int k = 0; k < kWStage; ++k) {
            const int e = k * kThreads + tid, v = e >> 1;
            const int hz = v / (kWHY * kWHX), r2 = v - hz * (kWHY * kWHX), hy = r2 / kWHX, hx = r2 - hy * kWHX;
            const int zz = z0 - 1 + hz, yy = y0 - 1 + hy, xx = x0 - 1 + hx;
            const bool in = ci0 + (e & 1) * 8 < cin && (unsigned)zz < (unsigned)w.D && (unsigned)yy < (unsigned)w.H &&
                            (unsigned)xx < (unsigned)w.W;
            const size_t at = in ? (((size_t)(zz >> shift) * Hs + (yy >> shift)) * Ws + (xx >> shift)) * cs + (e & 1) * 8 : 0;
            xcell[k] = load16(src + at);
            xin |= in ? 1u << k : 0u;
        }
#pragma unroll
        for (int k = 0; k < kGStage; ++k) {
            const int e = k * kThreads + tid;
            const int v = e / (2 * NT), c = e - v * (2 * NT);
            const int z = z0 + v / (kWY * kWX), y = y0 + (v / kWX) % kWY, x = x0 + v % kWX;
            const bool in = z < w.D && y < w.H && x < w.W;
            const size_t at = in ? (((size_t)z * w.H + y) * w.W + x) * w.cout + c * 8 : 0;
            gcell[k] = load16(w.gy + at);
            gin |= in ? 1u << k : 0u;
        }
    };
    load_brick(blockIdx.x);   // the host launches at most one workgroup per brick
    for (int b = blockIdx.x; b < w.bricks; b += gridDim.x) {
        __syncthreads();   // the previous brick's reads are done
#pragma unroll
        for (int k = 0; k < kWStage; ++k)
            if (k * kThreads + tid < kWHalo * 2) xs[k * kThreads + tid] = xin >> k & 1u ? xcell[k] : zero4;
#pragma unroll
        for (int k = 0; k < kGStage; ++k) {
            const int e = k * kThreads + tid;
            const int v = e / (2 * NT), c = e - v * (2 * NT);
            gs[((c >> 1) * kWVoxels + v) * 2 + (c & 1)] = gin >> k & 1u ? gcell[k] : zero4;
        }
        __syncthreads();
        if (b + (int)gridDim.x < w.bricks) load_brick(b + gridDim.x);
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

// Weights in the order conv3_brick_kernel's lanes read them: per 16 input
// channels, 16 output channels and step (dz, f) the 64 lanes' 8 values.
// transposed: the flipped, transposed weights of the backward-data pass (w
// stays [wco][27][wci], input channels are its wco).
__global__ void pack_weights_kernel(const float* w, int wci, int cin, int cout, int transposed, uint16_t* wt)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= cin / 16 * (cout / 16) * kConvFrags * 512) return;
    const int e = i & 7, lane = (i >> 3) & 63, frag = (i >> 9) % kConvFrags, tile = (i >> 9) / kConvFrags;
    const int co = tile % (cout / 16) * 16 + (lane & 15), kg = lane >> 4;
    const int ci = tile / (cout / 16) * 16 + (kg & 1) * 8 + e;
    const int dz = frag / 5, f = frag % 5, second = kg >> 1;
    // F1: row f, dx 0 or 1; P: dx 2, rows 0 and 1; Q: dx 2, rows 1 and 2
    const int dy = f < 3 ? f : f - 3 + second, dx = f < 3 ? second : 2;
    const int tap = (dz * 3 + dy) * 3 + dx;
    float v = transposed ? w[((size_t)ci * 27 + (26 - tap)) * wci + co] : w[((size_t)co * 27 + tap) * wci + ci];
    if (f >= 3 && dy == 1) v *= 0.5f;   // (in P and in Q)
    wt[i] = f2bf(v);
}

// The first layer's [16][27][2] weights in conv3_first_kernel's order.
__global__ void pack_first_weights_kernel(const float* w, uint16_t* wt)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 3 * 512) return;
    const int e = i & 7, lane = (i >> 3) & 63, row = (i >> 9) * 4 + (lane >> 4), dx = e >> 1;
    wt[i] = row < 9 && dx < 3 ? f2bf(w[((lane & 15) * 27 + row * 3 + dx) * 2 + (e & 1)]) : (uint16_t)0;
}

// g = (g + its parent's g_low / 8) where the activation y is positive, eight
// channels a thread
__global__ void join_gradients_kernel(const uint16_t* gl, int D, int H, int W, int C, const uint16_t* y, uint16_t* g)
{
    const int groups = C / 8;
    const size_t n = (size_t)D * H * W * groups;
    const int Hl = H / 2, Wl = W / 2;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const size_t m = i / groups;
        const int c = (int)(i - m * groups) * 8;
        const int z = (int)(m / ((size_t)W * H)), r = (int)(m - (size_t)z * W * H), yy = r / W, x = r - yy * W;
        const u32x4 low = load16(gl + (((size_t)(z / 2) * Hl + yy / 2) * Wl + x / 2) * C + c);
        const u32x4 act = load16(y + m * C + c);
        u32x4 v = load16(g + m * C + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float a, b, la, lb;
            dev::BF16::unpack2(v[e], a, b);
            dev::BF16::unpack2(low[e], la, lb);
            v[e] = gated(dev::BF16::pack2(a + la * 0.125f, b + lb * 0.125f), act[e]);
        }
        *reinterpret_cast<u32x4*>(g + m * C + c) = v;
    }
}

__global__ void pack_input_kernel(const float* x, float scale, const float* d, float dscale, size_t n, uint16_t* y)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const uint32_t a = f2bf(x[i] * scale), b = d ? f2bf(d[i] * dscale) : 0u;
        *reinterpret_cast<u32x4*>(y + 8 * i) = u32x4{a | (b << 16), 0u, 0u, 0u};
    }
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

// g_d1 = g_pred hw where d1 is positive; per block the sums of g_pred d1[c] and
// of g_pred: over each wave's lanes, then over its waves, in a fixed order
__global__ void __launch_bounds__(kThreads) head_backward_kernel(const uint16_t* d1, const float* gp, const float* hw,
                                                                 size_t n, uint16_t* gd1, float* partial)
{
    __shared__ float red[kThreads / 64][17];
    float s[17], h[16];
#pragma unroll
    for (int c = 0; c < 17; ++c) s[c] = 0.0f;
#pragma unroll
    for (int c = 0; c < 16; ++c) h[c] = hw[c];
    for (size_t m = (size_t)blockIdx.x * blockDim.x + threadIdx.x; m < n; m += (size_t)gridDim.x * blockDim.x) {
        const float g = gp[m];
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const u32x4 act = load16(d1 + m * 16 + half * 8);
            u32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int c = half * 8 + 2 * e;
                float a, b;
                dev::BF16::unpack2(act[e], a, b);
                s[c] += g * a;
                s[c + 1] += g * b;
                v[e] = gated(dev::BF16::pack2(g * h[c], g * h[c + 1]), act[e]);
            }
            *reinterpret_cast<u32x4*>(gd1 + m * 16 + half * 8) = v;
        }
        s[16] += g;
    }
#pragma unroll
    for (int c = 0; c < 17; ++c) {
        float t = s[c];
#pragma unroll
        for (int w = 32; w > 0; w /= 2) t += __shfl_xor(t, w);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x / 64][c] = t;
    }
    __syncthreads();
    if (threadIdx.x < 17) {
        float t = 0.0f;
        for (int q = 0; q < kThreads / 64; ++q) t += red[q][threadIdx.x];
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

namespace {
int conv_bricks(int D, int H, int W, int* nbx, int* nby)
{
    *nbx = (W + kBX - 1) / kBX;
    *nby = (H + kBY - 1) / kBY;
    return *nbx * *nby * ((D + kBZ - 1) / kBZ);
}

// one workgroup per brick, as many on every XCD
unsigned brick_groups(int bricks) { return (unsigned)((bricks + kXcds - 1) / kXcds * kXcds); }

template <Epilogue kEpi>
void launch_conv(const ConvArgs& a, hipStream_t stream)
{
    int nbx, nby;
    const int bricks = conv_bricks(a.D, a.H, a.W, &nbx, &nby);
    const unsigned groups = brick_groups(bricks);
    // 32 channels a workgroup share one halo, 16 give twice the workgroups:
    // those where 32 would leave CUs idle
    if (a.cout % 32 == 0 && bricks * (a.cout / 32) >= 512)
        conv3_brick_kernel<2, kEpi><<<dim3(groups, a.cout / 32), kConvThreads * 2, 0, stream>>>(a, nbx, nby, bricks);
    else
        conv3_brick_kernel<1, kEpi><<<dim3(groups, a.cout / 16), kConvThreads, 0, stream>>>(a, nbx, nby, bricks);
}
}  // namespace

void conv3_forward(const ConvArgs& a, hipStream_t stream)
{
    if (a.src.ca < 16 || (a.src.ca % 16) || (a.src.cb % 16)) fail("conv3: input channels must be multiples of 16");
    if (a.cout < 16 || a.cout % 16) fail("conv3: output channels must be a multiple of 16");
    if ((a.src.a_half || a.pool || a.children) && ((a.D | a.H | a.W) & 1)) fail("conv3: halved volumes need even sizes");
    if (a.head && a.cout != 16) fail("conv3: the head follows 16 channels");
    if (a.head) {
        int nbx, nby;
        const int bricks = conv_bricks(a.D, a.H, a.W, &nbx, &nby);
        conv3_brick_kernel<1, kHead><<<brick_groups(bricks), kConvThreads, 0, stream>>>(a, nbx, nby, bricks);
    } else if (a.pool) {
        launch_conv<kPool>(a, stream);
    } else if (a.children) {
        launch_conv<kChildren>(a, stream);
    } else {
        launch_conv<kStore>(a, stream);
    }
    hip_check(hipGetLastError(), "conv3 forward launch");
}

void conv3_first(const float* x, float scale, const float* d, float dscale, int D, int H, int W, const uint16_t* wt,
                 const float* bias, uint16_t* out, hipStream_t stream)
{
    int nbx, nby;
    const int bricks = conv_bricks(D, H, W, &nbx, &nby);
    conv3_first_kernel<<<brick_groups(bricks), kThreads, 0, stream>>>(x, scale, d, dscale, D, H, W, wt, bias, out, nbx, nby, bricks);
    hip_check(hipGetLastError(), "conv3 first layer launch");
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
    // (16 input channels a workgroup, all of them from a or from b)
    if (cout % 16 || cout > kMaxCout || cout == 48 || src.ca % (src.cb ? 16 : 8) || src.cb % 8 || cin > src.ca + src.cb)
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

void pack_weights(const float* w, int wci, int cin, int cout, bool transposed, uint16_t* wt, hipStream_t stream)
{
    const size_t n = conv_weight_count(cin, cout);
    pack_weights_kernel<<<(unsigned)((n + kThreads - 1) / kThreads), kThreads, 0, stream>>>(w, wci, cin, cout, transposed,
                                                                                           wt);
    hip_check(hipGetLastError(), "weight packing launch");
}

void pack_first_weights(const float* w, uint16_t* wt, hipStream_t stream)
{
    pack_first_weights_kernel<<<(kFirstWeights + kThreads - 1) / kThreads, kThreads, 0, stream>>>(w, wt);
    hip_check(hipGetLastError(), "weight packing launch");
}

void join_gradients(const uint16_t* g_low, int D, int H, int W, int C, const uint16_t* y, uint16_t* g,
                    hipStream_t stream)
{
    join_gradients_kernel<<<grid_for((size_t)D * H * W * C / 8), kThreads, 0, stream>>>(g_low, D, H, W, C, y, g);
}

void pack_input(const float* x, float scale, const float* d, float dscale, size_t count, uint16_t* y,
                hipStream_t stream)
{
    pack_input_kernel<<<grid_for(count), kThreads, 0, stream>>>(x, scale, d, dscale, count, y);
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
