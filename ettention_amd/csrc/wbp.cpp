#include "wbp.hpp"

#include <algorithm>

#include "geometry.hpp"

namespace etn {

namespace {

// NumericalAlgorithms::nearestPowerOfTwo (NumericalAlgorithms.cpp:20-31)
uint32_t next_power_of_two(uint32_t v)
{
    v--;
    v |= v >> 1;
    v |= v >> 2;
    v |= v >> 4;
    v |= v >> 8;
    v |= v >> 16;
    return v + 1;
}

}  // namespace

std::vector<float> WeightedBackProjection::ramLakKernel(uint32_t resolution)
{
    const float pi = 3.14159265358979323846f;
    const float pi2 = pi * pi;   // M_PI_F * M_PI_F, a float product
    std::vector<float> k(resolution);
    for (uint32_t i = 0; i < resolution; ++i) {
        const int position = (int)i - (int)(resolution / 2);
        if (position == 0) k[i] = 1.0f / 4.0f;
        else if (position % 2 == 0) k[i] = 0.0f;
        else k[i] = -1.0f / ((float)(position * position) * pi2);
    }
    return k;
}

dev::RampFilterParams WeightedBackProjection::filterParams(uint32_t nu, uint32_t nv, uint32_t taps)
{
    if (taps == 0 || taps % 2) fail("the ramp filter needs an even, non-zero number of taps");
    dev::RampFilterParams p{};
    p.nu = nu;
    p.nv = nv;
    // ConvolutionFourierSpaceImplementation::getUnifiedResolution: the larger
    // of filter (taps x 1) and image, rounded up to powers of two
    p.ux = next_power_of_two(std::max(taps, nu));
    p.uy = next_power_of_two(std::max(1u, nv));
    p.pad_x = ((int32_t)p.ux - (int32_t)nu) / 2;
    p.pad_y = ((int32_t)p.uy - (int32_t)nv) / 2;
    p.end_x = ((int32_t)p.ux + (int32_t)nu) / 2;
    p.end_y = ((int32_t)p.uy + (int32_t)nv) / 2;
    p.crop_x = (int32_t)(p.ux / 2) - (int32_t)(nu / 2);
    p.crop_y = (int32_t)(p.uy / 2) - (int32_t)(nv / 2);
    p.taps = taps;
    if (p.ux > dev::kMaxRampRow)
        unsupported("ramp filter: detector rows longer than " + std::to_string(dev::kMaxRampRow / 2) +
                    " pixels are not supported");
    return p;
}

WeightedBackProjection::WeightedBackProjection(const etn_reconstruction_desc& d, hipStream_t stream)
    : count_(d.projection_count), lambda_(d.lambda), projections_(static_cast<const float*>(d.projections))
{
    if (d.projection_count == 0 || (!d.tilt_angles && !d.geometries)) fail("No projections given!");
    if (!d.projections) fail("projection stack device pointer is null");
    if (d.flags & ETN_RECON_FLAG_16BIT_PROJECTIONS) unsupported("WBP filters f32 projections");
    const uint32_t nu = d.base_geometry.resolution[0], nv = d.base_geometry.resolution[1];
    if (nu == 0 || nv == 0) fail("detector resolution is zero");
    pixels_ = (size_t)nu * nv;
    params_ = filterParams(nu, nv, kFilterSize);

    geometries_ = projection_geometries(d);

    if (stream) {
        stream_ = stream;
    } else {
        ETN_HIP(hipStreamCreate(&stream_));
        own_stream_ = true;
    }
    etn_volume_geometry vg = d.volume;
    if (vg.subvolume_count == 0) vg.subvolume_count = 1;
    volume_ = std::make_unique<GpuVolume>(vg, d.voxel_type);
    volume_->fill(d.init_value, stream_);
    setup_ = std::make_unique<GeometricSetup>(geometries_[0], &volume_->properties());
    backward_ = std::make_unique<BackProjectionOperator>(setup_.get(), volume_.get(), &mask_, lambda_,
                                                         d.bp_samples ? d.bp_samples : 1, stream_);
    images_.allocate(2 * pixels_ * sizeof(float));
    filtered_ = {images_.as<float>(), nu, nv};
    length_ = {images_.as<float>() + pixels_, nu, nv};
    ray_length_ = std::make_unique<ComputeRayLengthKernel>(setup_.get(), &length_, stream_);
    const std::vector<float> k = ramLakKernel(kFilterSize);
    taps_.allocate(k.size() * sizeof(float));
    ETN_HIP(hipMemcpyAsync(taps_.get(), k.data(), taps_.bytes(), hipMemcpyHostToDevice, stream_));
    ETN_HIP(hipStreamSynchronize(stream_));
    slots_ = chunkSize();
    if ((d.flags & (ETN_RECON_FLAG_GENERIC_KERNELS | ETN_RECON_FLAG_EXACT_ARITHMETIC)) == 0) {
        // the sweep takes every projection or none; the whole volume is one slab
        const uint32_t samples = d.bp_samples ? d.bp_samples : 1;
        std::vector<dev::BackView> views(geometries_.size());
        const VolumeProperties whole = wholeVolume();
        // a sweep costs each workgroup 4.5 us a projection however small its tile is;
        // volumes of one tile that the fused passes' rows divide evenly take those for
        // many projections (121 of 32^3 493 us, 553 in sweeps; 16 of 32^3 140 / 85,
        // 121 of 24^3 567 / 543, of 32 x 32 x 128 1235 / 557)
        const uint32_t nx = whole.nx();
        const bool tiny = nx <= 32 && (nx & (nx - 1)) == 0 && nx % 4 == 0 && whole.nz() <= 32 && count_ > 40;
        bool sweep = samples == 1 && (d.flags & ETN_RECON_FLAG_LDS_BACK_PROJECTION) == 0 && !tiny;
        if (sweep) chunk_.allocate(sizeof(float) * 2 * pixels_ * slots_);
        for (size_t i = 0; sweep && i < views.size(); ++i) {
            const float* image = chunk_.as<float>() + 2 * pixels_ * (i % slots_);
            sweep = dev::make_back_view(make_slab_params(whole, 0),
                                        make_bp_params(geometries_[i], whole, samples, lambda_ / (float)count_), image,
                                        image + pixels_, &views[i]);
        }
        if (sweep) {
            const dev::SlabParams slab = make_slab_params(whole, 0);
            // rows whose rays lie inside the volume in y at every tilt
            std::vector<uint8_t> rows(nv, 1);
            for (const ParallelScannerGeometry& g : geometries_) {
                const std::vector<uint8_t> one = dev::row_classes(slab, make_ray_params(g, 1));
                for (uint32_t r = 0; r < nv; ++r) rows[r] = rows[r] && one[r];
            }
            groups_ = dev::sweep_groups(slab, views.data(), (int)views.size(), nv, rows);
            sweep = groups_.count > 0;
        }
        if (sweep) {
            views_.allocate(sizeof(dev::BackView) * views.size());
            ETN_HIP(hipMemcpyAsync(views_.get(), views.data(), views_.bytes(), hipMemcpyHostToDevice, stream_));
            ETN_HIP(hipStreamSynchronize(stream_));
        } else {
            chunk_.release();
            fused_ = FusedBackProjector::create(volume_.get(), geometries_, nu, nv, samples,
                                                (d.flags & ETN_RECON_FLAG_LDS_BACK_PROJECTION) != 0, stream_);
        }
    }
    if (usesFusedPath()) {
        std::vector<dev::RayParams> geo;
        for (const ParallelScannerGeometry& g : geometries_) geo.push_back(make_ray_params(g, 1));
        rays_.allocate(sizeof(dev::RayParams) * std::max<size_t>(geo.size(), 1));
        ETN_HIP(hipMemcpyAsync(rays_.get(), geo.data(), sizeof(dev::RayParams) * geo.size(), hipMemcpyHostToDevice,
                               stream_));
        ETN_HIP(hipStreamSynchronize(stream_));
    }
}

WeightedBackProjection::~WeightedBackProjection()
{
    if (stream_) (void)hipStreamSynchronize(stream_);
    if (own_stream_) (void)hipStreamDestroy(stream_);
}

void WeightedBackProjection::filter(const float* src, float* dst)
{
    dev::launch_ramp_filter(params_, taps_.as<float>(), src, dst, stream_);
}

// The volume as one slab: its slabs are contiguous in z, and a back projection
// treats every voxel alone.
VolumeProperties WeightedBackProjection::wholeVolume() const
{
    etn_volume_geometry g{};
    const VolumeProperties& v = volume_->properties();
    g.resolution[0] = v.nx();
    g.resolution[1] = v.ny();
    g.resolution[2] = v.nz();
    v.bbox_min().store(g.bbox_min);
    v.bbox_max().store(g.bbox_max);
    g.subvolume_count = 1;
    return VolumeProperties(g);
}

uint32_t WeightedBackProjection::chunkSize() const
{
    const size_t fit = kChunkBytes / (sizeof(float) * 2 * pixels_);
    return std::max(1u, std::min(count_, (uint32_t)std::min<size_t>(kChunk, std::max<size_t>(fit, 8))));
}

// Filtered images and ray lengths of projections first .. first + count - 1
// into the slots of chunk_, one launch each (one launch per image had cost 13
// and 4 us each, most of it launch and ramp-up).
void WeightedBackProjection::filterChunk(uint32_t first, uint32_t count)
{
    const VolumeProperties& vp = setup_->getVolume();
    float bmin[3], bmax[3];
    vp.bbox_min().store(bmin);
    vp.bbox_max().store(bmax);
    dev::launch_ramp_filter_batch(params_, taps_.as<float>(), projections_ + (size_t)first * pixels_, pixels_,
                                  chunk_.as<float>(), 2 * pixels_, count, stream_);
    dev::launch_ray_length_batch(bmin, bmax, rays_.as<dev::RayParams>() + first, count, params_.nu, params_.nv,
                                 chunk_.as<float>() + pixels_, 2 * pixels_, stream_);
}

void WeightedBackProjection::run() { runNiterations(count_); }

void WeightedBackProjection::runNiterations(uint32_t n)
{
    if (n > count_) fail("WBP: more projections requested than the stack holds");
    if (views_.get()) {
        // filtered images and ray lengths of a chunk of projections, then
        // their back projections in stack order in one sweep of the volume
        const dev::SlabParams slab = make_slab_params(wholeVolume(), 0);
        for (uint32_t i0 = 0; i0 < n; i0 += slots_) {
            const uint32_t k = std::min(n - i0, slots_);
            filterChunk(i0, k);
            hipEvent_t ev[2] = {nullptr, nullptr};
            if (launch_ms_) {
                for (auto& e : ev) ETN_HIP(hipEventCreate(&e));
                ETN_HIP(hipEventRecord(ev[0], stream_));
            }
            dev::sweep_back_project(slab, groups_, views_.as<dev::BackView>() + i0, (int)k, params_.nu, params_.nv,
                                    volume_->voxel_type(), volume_->data(), stream_);
            if (launch_ms_) {
                ETN_HIP(hipEventRecord(ev[1], stream_));
                ETN_HIP(hipEventSynchronize(ev[1]));
                float ms = 0.0f;
                ETN_HIP(hipEventElapsedTime(&ms, ev[0], ev[1]));
                launch_ms_->push_back(ms);
                for (auto& e : ev) (void)hipEventDestroy(e);
            }
        }
        return;
    }
    if (fused_) {
        // the same chunks, eight projections per volume sweep
        if (!chunk_.get()) chunk_.allocate(sizeof(float) * 2 * pixels_ * slots_);
        for (uint32_t i0 = 0; i0 < n; i0 += slots_) {
            std::vector<uint32_t> idx;
            std::vector<const float*> res, len;
            const uint32_t i1 = std::min(n, i0 + slots_);
            filterChunk(i0, i1 - i0);
            for (uint32_t i = i0; i < i1; ++i) {
                float* f = chunk_.as<float>() + 2 * pixels_ * (i - i0);
                idx.push_back(i);
                res.push_back(f);
                len.push_back(f + pixels_);
            }
            // backProject synchronises the stream before it returns, so the
            // next chunk may reuse the buffer
            fused_->backProject(idx, res, len, lambda_ / (float)count_, stream_, launch_ms_);
        }
        return;
    }
    for (uint32_t i = 0; i < n; ++i) {
        setup_->setScannerGeometry(geometries_[i]);
        filter(projections_ + (size_t)i * pixels_, filtered_.data);
        ray_length_->run();
        backward_->setInput(&filtered_, &length_, count_);
        backward_->execute();
        backward_->setInput(nullptr, nullptr, 1);
    }
}

void WeightedBackProjection::synchronize() { ETN_HIP(hipStreamSynchronize(stream_)); }

double WeightedBackProjection::timeKernels(int* kernel, uint32_t* launches)
{
    std::vector<float> ms;
    if (usesFusedPath()) {
        *kernel = views_.get() ? 3 : 0;
        launch_ms_ = &ms;
        try {
            run();
        } catch (...) {
            launch_ms_ = nullptr;
            throw;
        }
        launch_ms_ = nullptr;
    } else {
        *kernel = 2;
        hipEvent_t a, b;
        ETN_HIP(hipEventCreate(&a));
        ETN_HIP(hipEventCreate(&b));
        for (uint32_t i = 0; i < count_; ++i) {
            setup_->setScannerGeometry(geometries_[i]);
            filter(projections_ + (size_t)i * pixels_, filtered_.data);
            ray_length_->run();
            backward_->setInput(&filtered_, &length_, count_);
            ETN_HIP(hipEventRecord(a, stream_));
            backward_->execute();
            ETN_HIP(hipEventRecord(b, stream_));
            backward_->setInput(nullptr, nullptr, 1);
            ETN_HIP(hipEventSynchronize(b));
            float t = 0.0f;
            ETN_HIP(hipEventElapsedTime(&t, a, b));
            ms.push_back(t);
        }
        (void)hipEventDestroy(a);
        (void)hipEventDestroy(b);
    }
    *launches = (uint32_t)ms.size();
    double total = 0.0;
    for (float t : ms) total += t;
    return ms.empty() ? 0.0 : total / ms.size();
}

}  // namespace etn
