// Kernels of the learned correction network (3-D U-Net): bf16 activations in
// [D][H][W][C] order, 3x3x3 convolutions as implicit GEMMs on the gfx950
// matrix cores (v_mfma_f32_16x16x32_bf16, FP32 accumulation), and the
// elementwise / reduction kernels of training.  No reference counterpart.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace etn {
namespace nn {

// Input of a convolution: channels [0, ca) from `a` (at half resolution,
// read through nearest-neighbour upsampling, when a_half), then channels
// [ca, ca + cb) from `b` at full resolution.
struct ConvSrc {
    const uint16_t* a = nullptr;
    int ca = 0;
    int a_half = 0;
    const uint16_t* b = nullptr;
    int cb = 0;
};

// k steps of a convolution over 16 input channels (27 taps, two per step at most)
constexpr int kConvFrags = 15;
// packed weights of cin -> cout channels (multiples of 16); of the first layer
inline size_t conv_weight_count(int cin, int cout) { return (size_t)(cin / 16) * (cout / 16) * kConvFrags * 512; }
constexpr int kFirstWeights = 3 * 512;

struct ConvArgs {
    ConvSrc src;                  // channel counts are multiples of 16
    int D = 0, H = 0, W = 0;      // output size (full resolution of the input)
    const uint16_t* wt = nullptr; // pack_weights
    const float* bias = nullptr;  // [cout] or null
    int cout = 0;                 // a multiple of 16
    int relu = 0;
    uint16_t* out = nullptr;      // [D][H][W][cout] bf16
    const uint16_t* gate = nullptr;   // like out (children: half resolution): the result is 0 where gate <= 0
    uint16_t* pool = nullptr;     // [D/2][H/2][W/2][cout]: 2 x 2 x 2 averages of out
    int children = 0;             // out is [D/2][H/2][W/2][cout]: sums over 2 x 2 x 2 voxels (adjoint of upsampling)
    // the 1 x 1 x 1 head after 16 channels (weights [16], then the bias):
    // pred = x scale + head, unscaled back to x + head / scale when unscale; out may be null
    const float* head = nullptr;
    const float* x = nullptr;
    float scale = 1.0f;
    float* pred = nullptr;
    int unscale = 0;
};

// y = act(conv3(src) + bias)
void conv3_forward(const ConvArgs& a, hipStream_t stream);
// out[m][16] = relu(conv3(x scale, d dscale) + bias); d may be null (zeros); wt: pack_first_weights
void conv3_first(const float* x, float scale, const float* d, float dscale, int D, int H, int W, const uint16_t* wt,
                 const float* bias, uint16_t* out, hipStream_t stream);
// dw[co][tap][ci] = sum over voxels of gy[m][co] x[m + d(tap)][ci] for the
// first cin input channels, db[co] = sum over voxels of gy[m][co] (fp32);
// partial: wgrad_partial_floats(..., src.ca + src.cb, cout) floats of scratch
size_t wgrad_partial_floats(int D, int H, int W, int cin, int cout);
void conv3_weight_grad(const ConvSrc& src, int D, int H, int W, const uint16_t* gy, int cin, int cout, float* partial,
                       float* dw, float* db, hipStream_t stream);

// fp32 master weights w[co][27][ci] as bf16 in conv3_forward's order; wci: w's
// row length.  transposed: the flipped, transposed weights of the backward-data
// pass (conv cin = w's co, cout of w's ci from w on).
void pack_weights(const float* w, int wci, int cin, int cout, bool transposed, uint16_t* wt, hipStream_t stream);
void pack_first_weights(const float* w, uint16_t* wt, hipStream_t stream);

// g[m][c] = y[m][c] > 0 ? g[m][c] + g_low[parent(m)][c] / 8 : 0 (adjoint of the average pooling, then of the ReLU)
void join_gradients(const uint16_t* g_low, int D, int H, int W, int C, const uint16_t* y, uint16_t* g,
                    hipStream_t stream);

// y[m] = (x[m] scale, d[m] dscale, 0, 0, 0, 0, 0, 0) as eight bf16 channels; d may be null (zeros)
void pack_input(const float* x, float scale, const float* d, float dscale, size_t count, uint16_t* y,
                hipStream_t stream);
// r = pred - target * scale; partial sums of r^2 (fp64), g_pred = 2 r / voxels
void mse_loss(const float* pred, const float* target, float scale, size_t voxels, float* g_pred, double* partial,
              double* loss, hipStream_t stream);
// g_d1[m][c] = d1[m][c] > 0 ? g_pred[m] hw[c] : 0; partial head gradients (fp32) reduced into ghw[16], ghb[1]
void head_backward(const uint16_t* d1, const float* g_pred, const float* hw, size_t voxels, uint16_t* g_d1,
                   float* partial, float* ghw_ghb, hipStream_t stream);
void adam_step(float* p, const float* g, float* m, float* v, size_t count, float lr, float beta1, float beta2,
               float eps, float bc1, float bc2, hipStream_t stream);

}  // namespace nn
}  // namespace etn
