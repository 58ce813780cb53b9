#include "unet.hpp"

#include <algorithm>
#include <cmath>

namespace etn {

namespace {

struct LayerSpec {
    const char* name;
    int cin, cout, level;
};

// c1a reads (x, d); c4a reads concat(upsample(c3b), c2b), c5a reads concat(upsample(c4b), c1b)
constexpr LayerSpec kLayers[] = {
    {"c1a", 2, 16, 0},  {"c1b", 16, 16, 0}, {"c2a", 16, 32, 1}, {"c2b", 32, 32, 1}, {"c3a", 32, 64, 2},
    {"c3b", 64, 64, 2}, {"c4a", 96, 32, 1}, {"c4b", 32, 32, 1}, {"c5a", 48, 16, 0}, {"c5b", 16, 16, 0},
};
constexpr int kLayerCount = 10;
constexpr int kHead = 16;
constexpr int kInputChannels = 8;   // (x, d) padded to one 16-byte channel group
// upsampled input channels of a layer (they come first)
constexpr int upsampled(int i) { return i == 6 ? 64 : i == 8 ? 32 : 0; }

}  // namespace

size_t UNet3D::parameterCount()
{
    size_t n = 0;
    for (const LayerSpec& l : kLayers) n += (size_t)l.cout * 27 * l.cin + l.cout;
    return n + kHead + 1;
}

UNet3D::UNet3D(int nx, int ny, int nz, hipStream_t stream) : stream_(stream)
{
    if (nx < 4 || ny < 4 || nz < 4 || nx % 4 || ny % 4 || nz % 4)
        fail("the correction network needs volume sizes that are multiples of 4");
    for (int l = 0; l < 3; ++l) {
        D_[l] = nz >> l;
        H_[l] = ny >> l;
        W_[l] = nx >> l;
    }
    size_t at = 0;
    for (const LayerSpec& s : kLayers) {
        Layer L{s.name, s.cin, s.cout, s.level, at, at + (size_t)s.cout * 27 * s.cin};
        at = L.b + s.cout;
        layers_.push_back(L);
    }
    head_ = at;
    const size_t P = parameterCount();
    params_.allocate(sizeof(float) * P);
    ETN_HIP(hipMemsetAsync(params_.get(), 0, sizeof(float) * P, stream_));
    for (const Layer& L : layers_) {
        // the first layer reads the fp32 volumes and has no input gradient
        wt_.emplace_back(sizeof(uint16_t) * (L.cin < 16 ? (size_t)nn::kFirstWeights : nn::conv_weight_count(L.cin, L.cout)));
        wb_.emplace_back(L.cin < 16 ? 0 : sizeof(uint16_t) * nn::conv_weight_count(L.cout, L.cin));
        act_.emplace_back(sizeof(uint16_t) * voxels(L.level) * L.cout);
    }
    pool1_.allocate(sizeof(uint16_t) * voxels(1) * 16);
    pool2_.allocate(sizeof(uint16_t) * voxels(2) * 32);
    packAll();
}

void UNet3D::setParameters(const float* host, size_t count)
{
    if (count != parameterCount()) fail("parameter count mismatch");
    ETN_HIP(hipMemcpyAsync(params_.get(), host, sizeof(float) * count, hipMemcpyHostToDevice, stream_));
    ETN_HIP(hipStreamSynchronize(stream_));
    packAll();
    adam_t_ = 0;
    if (training_) {
        ETN_HIP(hipMemsetAsync(adam_m_.get(), 0, adam_m_.bytes(), stream_));
        ETN_HIP(hipMemsetAsync(adam_v_.get(), 0, adam_v_.bytes(), stream_));
    }
}

void UNet3D::getParameters(float* host, size_t count) const
{
    if (count != parameterCount()) fail("parameter count mismatch");
    ETN_HIP(hipMemcpyAsync(host, params_.get(), sizeof(float) * count, hipMemcpyDeviceToHost, stream_));
    ETN_HIP(hipStreamSynchronize(stream_));
}

void UNet3D::packAll()
{
    for (int i = 0; i < kLayerCount; ++i) {
        const Layer& L = layers_[i];
        const float* w = params_.as<float>() + L.w;
        if (L.cin < 16) {
            nn::pack_first_weights(w, wt_[i].as<uint16_t>(), stream_);
            continue;
        }
        nn::pack_weights(w, L.cin, L.cin, L.cout, false, wt_[i].as<uint16_t>(), stream_);
        // the decoder's first layers: the upsampled channels' part, then the skip's
        const int up = upsampled(i);
        if (up) nn::pack_weights(w, L.cin, L.cout, up, true, wb_[i].as<uint16_t>(), stream_);
        nn::pack_weights(w + up, L.cin, L.cout, L.cin - up, true,
                         wb_[i].as<uint16_t>() + nn::conv_weight_count(L.cout, up), stream_);
    }
}

nn::ConvSrc UNet3D::layerInput(int i) const
{
    nn::ConvSrc s;
    switch (i) {
        case 0: s.a = xin_.as<uint16_t>(); s.ca = kInputChannels; break;
        case 2: s.a = pool1_.as<uint16_t>(); s.ca = 16; break;
        case 4: s.a = pool2_.as<uint16_t>(); s.ca = 32; break;
        case 6:
            s.a = layerOutput(5); s.ca = 64; s.a_half = 1;
            s.b = layerOutput(3); s.cb = 32;
            break;
        case 8:
            s.a = layerOutput(7); s.ca = 32; s.a_half = 1;
            s.b = layerOutput(1); s.cb = 16;
            break;
        default: s.a = layerOutput(i - 1); s.ca = layers_[i - 1].cout; break;
    }
    return s;
}

void UNet3D::forward(const float* x, const float* d, float scale, float dscale, float* pred, bool predict)
{
    const float* p = params_.as<float>();
    for (int i = 0; i < kLayerCount; ++i) {
        const Layer& L = layers_[i];
        if (i == 0) {
            nn::conv3_first(x, scale, d, dscale, D_[0], H_[0], W_[0], wt_[0].as<uint16_t>(), p + L.b,
                            act_[0].as<uint16_t>(), stream_);
            continue;
        }
        nn::ConvArgs a;
        a.src = layerInput(i);
        a.D = D_[L.level];
        a.H = H_[L.level];
        a.W = W_[L.level];
        a.wt = wt_[i].as<uint16_t>();
        a.bias = p + L.b;
        a.cout = L.cout;
        a.relu = 1;
        a.out = act_[i].as<uint16_t>();
        if (i == 1) a.pool = pool1_.as<uint16_t>();
        if (i == 3) a.pool = pool2_.as<uint16_t>();
        if (i == kLayerCount - 1) {
            if (predict) a.out = nullptr;   // only the backward pass reads it
            a.head = p + head_;
            a.x = x;
            a.scale = scale;
            a.pred = pred;
            a.unscale = predict;
        }
        nn::conv3_forward(a, stream_);
    }
}

void UNet3D::predict(const float* x, const float* d, float scale, float dscale, float* out)
{
    if (!(scale > 0.0f) || !std::isfinite(scale) || !std::isfinite(dscale)) fail("scales must be finite, scale > 0");
    forward(x, d, scale, dscale, out, true);
}

void UNet3D::ensureTraining()
{
    if (training_) return;
    const size_t P = parameterCount();
    grads_.allocate(sizeof(float) * P);
    adam_m_.allocate(sizeof(float) * P);
    adam_v_.allocate(sizeof(float) * P);
    ETN_HIP(hipMemsetAsync(adam_m_.get(), 0, adam_m_.bytes(), stream_));
    ETN_HIP(hipMemsetAsync(adam_v_.get(), 0, adam_v_.bytes(), stream_));
    const size_t m0 = voxels(0), m1 = voxels(1), m2 = voxels(2);
    const size_t h = sizeof(uint16_t);
    xin_.allocate(h * m0 * kInputChannels);
    pred_.allocate(sizeof(float) * m0);
    gpred_.allocate(sizeof(float) * m0);
    gd1_.allocate(h * m0 * 16);
    gtmp_.allocate(h * std::max({m0 * 16, m1 * 32, m2 * 64}));
    ge1_.allocate(h * m0 * 16);
    ge2_.allocate(h * m1 * 32);
    ge3_.allocate(h * m2 * 64);
    gd2_.allocate(h * m1 * 32);
    gp_.allocate(h * std::max(m2 * 32, m1 * 16));
    size_t wpart = 0;
    for (const Layer& L : layers_)
        wpart = std::max(wpart, nn::wgrad_partial_floats(D_[L.level], H_[L.level], W_[L.level],
                                                         std::max(L.cin, kInputChannels), L.cout));
    wpart_.allocate(sizeof(float) * wpart);
    hpart_.allocate(sizeof(float) * 1024 * 17);
    loss_.allocate(sizeof(double));
    lpart_.allocate(sizeof(double) * 1024);
    training_ = true;
}

void UNet3D::backward()
{
    float* g = grads_.as<float>();
    // layer i from its output's gradient gy (already zero where the ReLU is):
    // the parameters' gradients, and the input's in gx, zero where gate's ReLU
    // is; of a layer on upsampled channels, gx takes the skip's and gx_up the
    // upsampled volume's at its own resolution
    auto layer_back = [&](int i, const uint16_t* gy, uint16_t* gx, const uint16_t* gate, uint16_t* gx_up = nullptr,
                          const uint16_t* gate_up = nullptr) {
        const Layer& L = layers_[i];
        const int D = D_[L.level], H = H_[L.level], W = W_[L.level];
        nn::conv3_weight_grad(layerInput(i), D, H, W, gy, L.cin, L.cout, wpart_.as<float>(), g + L.w, g + L.b, stream_);
        if (!gx) return;
        nn::ConvArgs a;
        a.src.a = gy;
        a.src.ca = L.cout;
        a.D = D;
        a.H = H;
        a.W = W;
        a.wt = wb_[i].as<uint16_t>();
        const int up = upsampled(i);
        if (up) {
            a.cout = up;
            a.out = gx_up;
            a.gate = gate_up;
            a.children = 1;
            nn::conv3_forward(a, stream_);
            a.children = 0;
            a.wt += nn::conv_weight_count(L.cout, up);
        }
        a.cout = L.cin - up;
        a.out = gx;
        a.gate = gate;
        nn::conv3_forward(a, stream_);
    };
    uint16_t* gtmp = gtmp_.as<uint16_t>();
    uint16_t* gp = gp_.as<uint16_t>();
    uint16_t* gd1 = gd1_.as<uint16_t>();
    uint16_t* gd2 = gd2_.as<uint16_t>();
    uint16_t* ge1 = ge1_.as<uint16_t>();
    uint16_t* ge2 = ge2_.as<uint16_t>();
    uint16_t* ge3 = ge3_.as<uint16_t>();
    const float* p = params_.as<float>();
    nn::head_backward(layerOutput(9), gpred_.as<float>(), p + head_, voxels(0), gd1, hpart_.as<float>(), g + head_,
                      stream_);
    // decoder, full and half resolution (the skips' gradients stay without
    // their ReLU until the encoder's own arrive)
    layer_back(9, gd1, gtmp, layerOutput(8));
    layer_back(8, gtmp, ge1, nullptr, gd2, layerOutput(7));
    layer_back(7, gd2, gtmp, layerOutput(6));
    layer_back(6, gtmp, ge2, nullptr, ge3, layerOutput(5));
    // bottleneck
    layer_back(5, ge3, gtmp, layerOutput(4));
    layer_back(4, gtmp, gp, nullptr);
    nn::join_gradients(gp, D_[1], H_[1], W_[1], 32, layerOutput(3), ge2, stream_);
    // encoder, half and full resolution
    layer_back(3, ge2, gtmp, layerOutput(2));
    layer_back(2, gtmp, gp, nullptr);
    nn::join_gradients(gp, D_[0], H_[0], W_[0], 16, layerOutput(1), ge1, stream_);
    layer_back(1, ge1, gtmp, layerOutput(0));
    layer_back(0, gtmp, nullptr, nullptr);
}

double UNet3D::gradient(const float* x, const float* d, const float* target, float scale, float dscale)
{
    if (!(scale > 0.0f) || !std::isfinite(scale) || !std::isfinite(dscale)) fail("scales must be finite, scale > 0");
    ensureTraining();
    // the first layer's weight gradient reads its input as channels
    nn::pack_input(x, scale, d, dscale, voxels(0), xin_.as<uint16_t>(), stream_);
    forward(x, d, scale, dscale, pred_.as<float>(), false);
    nn::mse_loss(pred_.as<float>(), target, scale, voxels(0), gpred_.as<float>(), lpart_.as<double>(),
                 loss_.as<double>(), stream_);
    backward();
    double loss = 0.0;
    ETN_HIP(hipMemcpyAsync(&loss, loss_.get(), sizeof(double), hipMemcpyDeviceToHost, stream_));
    ETN_HIP(hipStreamSynchronize(stream_));
    return loss;
}

void UNet3D::copyGradient(float* host, size_t count) const
{
    if (!training_) fail("no gradient has been computed");
    if (count != parameterCount()) fail("parameter count mismatch");
    ETN_HIP(hipMemcpyAsync(host, grads_.get(), sizeof(float) * count, hipMemcpyDeviceToHost, stream_));
    ETN_HIP(hipStreamSynchronize(stream_));
}

double UNet3D::trainStep(const float* x, const float* d, const float* target, float scale, float dscale, float lr)
{
    const double loss = gradient(x, d, target, scale, dscale);
    ++adam_t_;
    const float b1 = 0.9f, b2 = 0.999f;
    const float bc1 = 1.0f - std::pow(b1, (float)adam_t_), bc2 = 1.0f - std::pow(b2, (float)adam_t_);
    nn::adam_step(params_.as<float>(), grads_.as<float>(), adam_m_.as<float>(), adam_v_.as<float>(), parameterCount(),
                  lr, b1, b2, 1e-8f, bc1, bc2, stream_);
    packAll();
    return loss;
}

double UNet3D::timeForward(const float* x, float scale, double* flops)
{
    double f = 0.0;
    for (const Layer& L : layers_) f += 2.0 * 27.0 * L.cin * L.cout * (double)voxels(L.level);
    f += 2.0 * kHead * (double)voxels(0);
    if (flops) *flops = f;
    if (!pred_.get()) pred_.allocate(sizeof(float) * voxels(0));
    hipEvent_t a, b;
    ETN_HIP(hipEventCreate(&a));
    ETN_HIP(hipEventCreate(&b));
    ETN_HIP(hipEventRecord(a, stream_));
    forward(x, nullptr, scale, 0.0f, pred_.as<float>(), true);
    ETN_HIP(hipEventRecord(b, stream_));
    ETN_HIP(hipEventSynchronize(b));
    float ms = 0.0f;
    ETN_HIP(hipEventElapsedTime(&ms, a, b));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    return ms;
}

}  // namespace etn
