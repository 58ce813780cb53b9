// WBP (plugins/WBPPlugin/src/reconstruction/WBP.cpp:13-84): weighted back
// projection, the other caller of the back-projection operator.  Every
// projection is ramp-filtered (GenerateRamLakKernel + ConvolutionOperator),
// its pixel-centre chord through the volume box becomes the ray length
// (ComputeRayLengthKernel), and it is back-projected with lambda / N.
#pragma once

#include <memory>
#include <vector>

#include "fused.hpp"
#include "kernels.hpp"
#include "operators.hpp"
#include "reconstruction.hpp"

namespace etn {

class WeightedBackProjection final : public ReconstructionAlgorithm {
public:
    static constexpr uint32_t kFilterSize = 128;   // WBP.cpp:30

    WeightedBackProjection(const etn_reconstruction_desc& desc, hipStream_t stream);
    ~WeightedBackProjection() override;

    // WBP::run: every projection once, in stack order.
    void run() override;
    // WBP::runNiterations: projections 0 .. n-1.
    void runNiterations(uint32_t n) override;
    void runSingleIteration() override { runNiterations(1); }
    GpuVolume* getReconstructedVolume() override { return volume_.get(); }
    void synchronize() override;
    hipStream_t stream() const override { return stream_; }
    // Single-axis tilt geometries back-project a chunk of up to kChunk projections
    // per volume sweep, or on the fused kernels eight (oversampled, the LDS back
    // projection), with fast arithmetic, unless the generic kernels or exact
    // arithmetic are asked for.
    bool usesFusedPath() const override { return fused_ != nullptr || views_.get() != nullptr; }
    // One more run() with HIP events around the back projections: the average
    // sweep (*kernel = 3), fused launch carrying eight projections (0) or
    // generic back projection (2).  Adds to the volume.
    double timeKernels(int* kernel, uint32_t* launches) override;

    // GenerateRamLakKernel.cl: value at position p = i - resolution / 2 is 1/4
    // at 0, 0 at even p, -1 / (p^2 pi^2) at odd p, in float.
    static std::vector<float> ramLakKernel(uint32_t resolution);
    // Filter parameters for an nu x nv image (ConvolutionFourierSpaceImplementation,
    // PaddingForFFT.cl, CroppingForFFT.cl).
    static dev::RampFilterParams filterParams(uint32_t nu, uint32_t nv, uint32_t taps);
    // ConvolutionOperator::execute on one device image.
    void filter(const float* src, float* dst);

private:
    // Projections of a chunk: their filtered images and ray lengths stay allocated
    // with the object, within kChunkBytes as long as that holds eight (64 of 1024^2,
    // 16 of 2048^2, 8 of 4096^2: 1 GiB).
    static constexpr uint32_t kChunk = 64;
    static constexpr size_t kChunkBytes = (size_t)512 << 20;
    uint32_t chunkSize() const;
    void filterChunk(uint32_t first, uint32_t count);
    VolumeProperties wholeVolume() const;

    hipStream_t stream_ = nullptr;
    bool own_stream_ = false;
    uint32_t count_;
    float lambda_;
    const float* projections_;
    size_t pixels_;
    std::vector<ParallelScannerGeometry> geometries_;
    std::unique_ptr<GpuVolume> volume_;
    GpuMask mask_;   // WBP passes no mask (WBP.cpp:45)
    std::unique_ptr<GeometricSetup> setup_;
    std::unique_ptr<BackProjectionOperator> backward_;
    DeviceBuffer images_;   // filtered projection + ray length
    DeviceImage filtered_, length_;
    std::unique_ptr<ComputeRayLengthKernel> ray_length_;
    DeviceBuffer taps_;
    dev::RampFilterParams params_;
    std::unique_ptr<FusedBackProjector> fused_;
    DeviceBuffer rays_;   // fused paths: every projection's ray geometry, for the batched ray lengths
    DeviceBuffer views_;  // sweep path: every projection's table entry (its images: a slot of chunk_)
    dev::SweepGroups groups_;
    uint32_t slots_ = 0;  // projections of a chunk
    DeviceBuffer chunk_;  // their filtered images and ray lengths
    std::vector<float>* launch_ms_ = nullptr;    // set while timeKernels runs
};

}  // namespace etn
