"""The fused kernels' register back projection against their LDS back
projection (ETN_RECON_FLAG_LDS_BACK_PROJECTION).

With fast arithmetic, nx a multiple of 4 and no oversampling, the fused
kernels apply a pass's back projections to each group of 4 voxels in
registers as the band arrives from HBM, all of them in block order, and stage
the detector records of every back projection of the pass once per launch
(in a 160 KiB LDS array when they do not fit the workgroup shape's own).  The
LDS path applies one back projection after another to the band in LDS and
restages the records per projection and band.  Every voxel sees the same
chain of updates and roundings on both, so the volumes must agree bit for
bit: single projections (SART), blocks of 4 and 8 (up to 8 back projections
per pass), long-object compensation, masks, 16-bit storage, both workgroup
shapes, several tiles, and the weighted back projection's many-projection
passes."""
import numpy as np
import pytest

import ettention_amd as E
from ettention_amd import api as A
from ettention_amd import synthetic as S

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

LDS = E.ETN_RECON_FLAG_LDS_BACK_PROJECTION


def inputs(shape, ntilts, seed, **kw):
    nx, ny, nz = shape
    vg = E.VolumeGeometry.make((nx, ny, nz))
    base = E.ScannerGeometry.mrc_base(nx, ny)
    tilts = np.linspace(-60.0, 60.0, ntilts).astype(np.float32)
    ph = S.ellipsoid_phantom((nz, ny, nx), seed=seed, device=torch.device("cuda"))
    projs = torch.zeros((ntilts, ny, nx), dtype=torch.float32, device="cuda")
    scratch = torch.zeros((ny, nx), dtype=torch.float32, device="cuda")
    for i, t in enumerate(tilts):
        scratch.zero_()
        A.forward_project(vg, ph, A.rotate(base, float(t)), projs[i], scratch)
    torch.cuda.synchronize()
    d = dict(volume=vg, base_geometry=base, tilt_angles=tilts, projections=S.add_gaussian_noise(projs, 0.02, seed=seed),
             algorithm="sart", lam=0.3, projection_iteration="random")
    d.update(kw)
    return d


def run(case, flags=0, threads=None, tile=None, iterations=2):
    r = A.BlockIterativeReconstructionOperator(flags=flags, **case)
    assert r.uses_fused_path()
    if threads is not None:
        r.set_workgroup_threads(threads)
    if tile is not None:
        r.set_tile(*tile)
    r.run_iterations(iterations)
    r.synchronize()
    return r.get_reconstructed_volume(dtype=torch.float32).cpu().numpy(), r.residual_norm()


FUSED, SWEEPING = 0, 3      # the library's own report of what it timed


def timed_kernel(case, flags=0):
    kernel, ms, launches = A.BlockIterativeReconstructionOperator(
        flags=flags | E.ETN_RECON_FLAG_NO_AUTOTUNE, **case).time_kernels()
    assert launches > 0 and (kernel != SWEEPING or ms > 0.0)   # (a single block has no steady fused pass)
    return kernel


CASES = {
    "sart": ((64, 64, 64), 41, {}),
    "block4": ((48, 48, 40), 61, dict(algorithm="blockiterative", block_size=4, projection_iteration="maxangle")),
    "block8": ((128, 64, 64), 61, dict(algorithm="blockiterative", block_size=8)),
    "sirt_loc": ((64, 32, 48), 21, dict(algorithm="sirt", use_long_object_compensation=True)),
    "block8_bf16": ((64, 64, 32), 41, dict(algorithm="blockiterative", block_size=8, voxel_type="bfloat16")),
    "sart_half": ((64, 48, 40), 31, dict(voxel_type="half")),
    # 512 wide: 8 record sets of 512-voxel rows no longer fit the workgroup
    # shape's LDS, so one-plane tiles take the 80 KiB register path (bands of
    # at most 7 rows) and wider tiles the 160 KiB one
    "block8_wide": ((512, 8, 24), 61, dict(algorithm="blockiterative", block_size=8)),
    "block8_wide_bf16": ((512, 8, 24), 41, dict(algorithm="blockiterative", block_size=8, voxel_type="bfloat16")),
}


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("threads", [512, 256])
def test_register_back_projection_equals_lds_back_projection(name, threads):
    shape, ntilts, kw = CASES[name]
    case = inputs(shape, ntilts, 7100 + len(name), **kw)
    print("register bp case", name, threads, flush=True)
    reg, reg_norm = run(case, threads=threads)
    lds, lds_norm = run(case, flags=LDS, threads=threads)
    np.testing.assert_array_equal(reg, lds)
    assert reg_norm == lds_norm


@pytest.mark.parametrize("name", ["sart", "block8", "block8_wide"])
def test_register_back_projection_with_a_mask(name):
    shape, ntilts, kw = CASES[name]
    nx, ny, nz = shape
    rng = np.random.default_rng(71)
    mask = torch.from_numpy(rng.integers(0, 256, (nz, ny, nx), dtype=np.uint8)).cuda()
    case = inputs(shape, ntilts, 7200, mask=mask, **kw)
    for threads in (512, 256):
        print("register bp mask case", name, threads, flush=True)
        reg, _ = run(case, threads=threads)
        lds, _ = run(case, flags=LDS, threads=threads)
        np.testing.assert_array_equal(reg, lds)


@pytest.mark.parametrize("tile", [(1, 1), (1, 5), (2, 3), (4, 2), (8, 1)])
def test_register_back_projection_every_tile(tile):
    # planes x band rows; every tile cuts the same work, on both paths
    shape, ntilts, kw = CASES["block4"]
    case = inputs(shape, ntilts, 7300, **kw)
    print("register bp tile", tile, flush=True)
    ref, _ = run(case, flags=LDS | E.ETN_RECON_FLAG_NO_AUTOTUNE)
    got, _ = run(case, flags=E.ETN_RECON_FLAG_NO_AUTOTUNE, tile=tile)
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("tile", [(1, 1), (1, 3), (1, 12), (2, 2), (4, 1)])
def test_register_back_projection_wide_tiles(tile):
    # 512 wide, 8 back projections per pass: one plane per tile takes the
    # 80 KiB register path with the band cut to what fits beside the records,
    # two planes the 160 KiB one, four (whose records exceed even that) the
    # LDS path
    shape, ntilts, kw = CASES["block8_wide"]
    case = inputs(shape, ntilts, 7500, **kw)
    print("register bp wide tile", tile, flush=True)
    ref, _ = run(case, flags=LDS | E.ETN_RECON_FLAG_NO_AUTOTUNE, threads=512)
    got, _ = run(case, flags=E.ETN_RECON_FLAG_NO_AUTOTUNE, threads=512, tile=tile)
    np.testing.assert_array_equal(got, ref)


def test_wbp_register_back_projection_equals_lds():
    # the weighted back projection's passes carry 8 projections each
    n = 64
    vg = E.VolumeGeometry.make((n, n, n))
    base = E.ScannerGeometry.mrc_base(n, n)
    tilts = np.linspace(-60.0, 60.0, 37).astype(np.float32)
    ph = S.ellipsoid_phantom((n, n, n), seed=7400, device=torch.device("cuda"))
    projs = torch.zeros((len(tilts), n, n), dtype=torch.float32, device="cuda")
    scratch = torch.zeros((n, n), dtype=torch.float32, device="cuda")
    for i, t in enumerate(tilts):
        scratch.zero_()
        A.forward_project(vg, ph, A.rotate(base, float(t)), projs[i], scratch)
    vols = []
    for flags in (0, LDS):
        for kw in (dict(), dict(bp_samples=9)):   # 9 samples: oversampled, the LDS path either way
            r = A.WeightedBackProjection(volume=vg, base_geometry=base, tilt_angles=tilts, projections=projs,
                                         lam=1.0, flags=flags, **kw)
            assert r.uses_fused_path()
            r.run()
            vols.append(r.get_reconstructed_volume().cpu().numpy())
    np.testing.assert_array_equal(vols[0], vols[2])
    np.testing.assert_array_equal(vols[1], vols[3])


# blocks as separate sweeps (the default) against the fused passes on the LDS
# back projection: nx off a multiple of 4, one and two planes a workgroup, both z
# directions, more projections in a block than in a sweep (other detectors, four
# planes and several rays a thread: test_gpu_sweep_geometries.py)
SWEEPS = [((135, 131, 120), 23, 8, 60.0, "float"), ((64, 522, 64), 9, 9, 60.0, "float"), ((300, 160, 180), 9, 4, 60.0, "float"),
          ((520, 70, 64), 19, 8, 60.0, "bfloat16"), ((136, 130, 120), 40, 0, 60.0, "half"), ((130, 130, 128), 30, 12, 150.0, "float")]


@pytest.mark.parametrize("shape,ntilts,block,reach,voxel", SWEEPS)
@pytest.mark.parametrize("loc", [False, True])
def test_block_sweeps_equal_the_fused_passes(shape, ntilts, block, reach, voxel, loc):
    nx, ny, nz = shape
    rng = np.random.default_rng(ntilts)
    case = dict(volume=E.VolumeGeometry.make(shape), base_geometry=E.ScannerGeometry.mrc_base(nx, ny),
                tilt_angles=np.linspace(-reach, reach, ntilts).astype(np.float32),
                projections=torch.from_numpy(rng.normal(1.0, 0.3, (ntilts, ny, nx)).astype(np.float32)).cuda(),
                algorithm="blockiterative" if block else "sirt", block_size=block, lam=0.3, voxel_type=voxel,
                use_long_object_compensation=loc)
    v, norm = run(case)
    w, ref = run(case, flags=LDS)
    np.testing.assert_array_equal(v, w)
    assert norm == ref


def test_time_kernels_tells_sweeps_from_fused_passes():
    # 16 projections in blocks of 8: per block one back sweep and a forward sweep
    # for each z direction among its projections
    shape = (130, 130, 128)
    case = dict(volume=E.VolumeGeometry.make(shape), base_geometry=E.ScannerGeometry.mrc_base(130, 130),
                tilt_angles=np.linspace(0, 60, 16).astype(np.float32),
                projections=torch.ones((16, 130, 130), device="cuda"), algorithm="blockiterative", block_size=8,
                projection_iteration="identity")
    kernel, ms, launches = A.BlockIterativeReconstructionOperator(**case).time_kernels()
    assert (kernel, launches) == (SWEEPING, 4) and ms > 0.0
    assert timed_kernel(case, LDS) == FUSED
    r = A.BlockIterativeReconstructionOperator(**case)
    r.set_tile(*r.tile())                       # a tile is one of the fused passes'
    assert r.time_kernels()[0] == FUSED


# the residual norm of a swept reconstruction runs in forward sweeps (of up to 8
# projections, both z directions in a chunk) and is the fused passes' bit for bit
@pytest.mark.parametrize("shape,block,fp,masked,voxel", [((130, 131, 140), 8, 1, False, "float"), ((97, 96, 96), 9, 1, True, "half"),
                                                         ((104, 80, 98), 2, 2, False, "bfloat16")])
def test_residual_norm_of_sweeps(shape, block, fp, masked, voxel):
    nx, ny, nz = shape
    rng = np.random.default_rng(block)
    case = dict(volume=E.VolumeGeometry.make(shape), base_geometry=E.ScannerGeometry.mrc_base(nx, ny),
                tilt_angles=np.linspace(-150, 150, 21).astype(np.float32),
                projections=torch.from_numpy(rng.normal(1.0, 0.3, (21, ny, nx)).astype(np.float32)).cuda(),
                algorithm="blockiterative", block_size=block, lam=0.3, voxel_type=voxel, fp_samples=fp,
                bp_samples=4 if fp > 1 else 1, skip_projections=(0, 7, 8), use_long_object_compensation=True)
    if masked:
        case["mask"] = torch.from_numpy(rng.integers(0, 256, (nz, ny, nx)).astype(np.uint8)).cuda()
    r = A.BlockIterativeReconstructionOperator(**case)
    r.run_iterations(1)
    norm = r.residual_norm()
    assert timed_kernel(case) == SWEEPING
    r.set_tile(*r.tile())
    assert norm == r.residual_norm() and norm > 0.0


# which reconstructions are swept: sizes on both sides of the lines that
# measurements drew (FusedEngineImpl::sweepsPay)
@pytest.mark.parametrize("shape,block,voxel,fp,bp,masked,kernel", [
    ((128, 160, 128), 8, "float", 1, 1, False, FUSED), ((128, 128, 132), 8, "float", 1, 1, False, SWEEPING),
    ((32, 512, 300), 8, "float", 1, 1, False, FUSED), ((48, 400, 300), 8, "float", 1, 1, False, SWEEPING),
    ((256, 256, 32), 8, "float", 1, 1, False, SWEEPING), ((512, 512, 8), 8, "float", 1, 1, False, FUSED),
    ((64, 512, 256), 8, "half", 1, 1, False, FUSED), ((112, 200, 200), 8, "half", 1, 1, False, SWEEPING),
    ((512, 256, 32), 8, "bfloat16", 1, 1, False, FUSED), ((512, 256, 48), 8, "bfloat16", 1, 1, False, SWEEPING),
    ((64, 256, 300), 16, "bfloat16", 1, 1, False, SWEEPING), ((128, 256, 256), 4, "float", 1, 1, False, FUSED),
    ((256, 512, 64), 4, "float", 1, 1, False, SWEEPING), ((256, 512, 64), 4, "bfloat16", 1, 1, False, FUSED),
    ((256, 512, 64), 6, "bfloat16", 1, 1, False, SWEEPING), ((32, 512, 64), 8, "float", 1, 1, True, FUSED),
    ((96, 96, 96), 8, "float", 1, 1, True, SWEEPING), ((96, 96, 96), 1, "float", 2, 4, False, FUSED),
    ((104, 104, 104), 1, "float", 2, 4, False, SWEEPING), ((132, 1000, 20), 1, "float", 1, 9, False, FUSED),
    ((200, 400, 32), 1, "float", 1, 4, False, FUSED), ((204, 204, 204), 1, "float", 2, 1, False, FUSED),
    ((204, 204, 204), 1, "float", 3, 1, False, SWEEPING),
    # estimates far apart, more than two rays a thread
    ((200, 69, 614), 4, "half", 1, 1, False, SWEEPING), ((32, 96, 512), 16, "float", 3, 9, False, SWEEPING),
    ((132, 1000, 20), 1, "bfloat16", 4, 9, True, FUSED), ((512, 96, 48), 1, "half", 3, 16, False, SWEEPING)])
def test_sweeps_where_they_pay(shape, block, voxel, fp, bp, masked, kernel):
    nx, ny, nz = shape
    case = dict(volume=E.VolumeGeometry.make(shape), base_geometry=E.ScannerGeometry.mrc_base(nx, ny),
                tilt_angles=np.linspace(-60, 60, 16).astype(np.float32),
                projections=torch.ones((16, ny, nx), device="cuda"), algorithm="blockiterative", block_size=block,
                voxel_type=voxel, fp_samples=fp, bp_samples=bp)
    if masked:
        case["mask"] = torch.full((nz, ny, nx), 255, dtype=torch.uint8, device="cuda")
    assert timed_kernel(case) == kernel


def test_wbp_time_kernels_tells_sweeps_from_fused_passes():
    n, count = 40, 70                           # two chunks of up to 64 projections, a sweep each
    case = dict(volume=E.VolumeGeometry.make((n, n, n)), base_geometry=E.ScannerGeometry.mrc_base(n, n),
                tilt_angles=np.linspace(-60, 60, count).astype(np.float32),
                projections=torch.ones((count, n, n), device="cuda"))
    assert A.WeightedBackProjection(**case).time_kernels()[::2] == (SWEEPING, 2)
    assert A.WeightedBackProjection(flags=LDS, **case).time_kernels()[0] == FUSED
    assert A.WeightedBackProjection(flags=E.ETN_RECON_FLAG_GENERIC_KERNELS, **case).time_kernels()[0] == 2


# sample patterns, sub-rays and masks in the sweeps, within what two
# reconstructions in single precision may differ by
@pytest.mark.parametrize("shape,ntilts,block,fp,bp,masked,voxel", [
    ((90, 81, 77), 17, 0, 1, 1, True, "float"), ((88, 83, 76), 13, 8, 1, 1, True, "half"),
    ((88, 81, 77), 9, 1, 2, 4, False, "float"), ((91, 82, 70), 9, 1, 4, 9, True, "float"),
    ((92, 81, 72), 12, 4, 3, 16, True, "float"), ((88, 80, 79), 9, 1, 1, 9, True, "bfloat16")])
def test_sampled_sweeps_match_the_fused_passes(shape, ntilts, block, fp, bp, masked, voxel):
    nx, ny, nz = shape
    rng = np.random.default_rng(ntilts)
    case = dict(volume=E.VolumeGeometry.make(shape), base_geometry=E.ScannerGeometry.mrc_base(nx, ny),
                tilt_angles=np.linspace(-60, 60, ntilts).astype(np.float32),
                projections=torch.from_numpy(rng.normal(1.0, 0.3, (ntilts, ny, nx)).astype(np.float32)).cuda(),
                algorithm="blockiterative" if block else "sirt", block_size=block, lam=0.3, voxel_type=voxel,
                fp_samples=fp, bp_samples=bp)
    if masked:
        mask = rng.integers(0, 256, (nz, ny, nx)).astype(np.uint8)
        mask[:, : ny // 3] = 0
        case["mask"] = torch.from_numpy(mask).cuda()
    v, norm = run(case)
    w, ref = run(case, flags=LDS)
    bound = 2e-5 if voxel == "float" else 1e-2
    assert np.linalg.norm(v - w) <= bound * np.linalg.norm(w)
    assert abs(norm - ref) <= bound * ref


# the same bit for bit, also with shapes that take two planes a workgroup (nx in
# fours and odd) and with a tile set between two iterations, which leaves the
# sweeps for the fused passes
@pytest.mark.parametrize("shape,ntilts,block,fp,bp,masked,voxel", [
    ((90, 81, 77), 17, 0, 1, 1, True, "float"), ((88, 83, 76), 13, 8, 1, 1, True, "half"),
    ((104, 81, 98), 9, 1, 2, 4, False, "float"), ((91, 82, 76), 9, 1, 4, 9, True, "float"),
    ((92, 81, 72), 12, 4, 3, 16, True, "float"), ((88, 80, 79), 9, 1, 1, 9, True, "bfloat16"),
    ((250, 300, 16), 5, 1, 4, 9, True, "bfloat16"), ((252, 300, 16), 5, 1, 4, 9, True, "float"),
    ((252, 260, 130), 3, 1, 3, 1, False, "half")])
def test_sampled_sweeps_equal_the_fused_passes(shape, ntilts, block, fp, bp, masked, voxel):
    nx, ny, nz = shape
    rng = np.random.default_rng(ntilts)
    case = dict(volume=E.VolumeGeometry.make(shape), base_geometry=E.ScannerGeometry.mrc_base(nx, ny),
                tilt_angles=np.linspace(-60, 60, ntilts).astype(np.float32),
                projections=torch.from_numpy(rng.normal(1.0, 0.3, (ntilts, ny, nx)).astype(np.float32)).cuda(),
                algorithm="blockiterative" if block else "sirt", block_size=block, lam=0.3, voxel_type=voxel,
                fp_samples=fp, bp_samples=bp)
    if masked:
        mask = rng.integers(0, 256, (nz, ny, nx)).astype(np.uint8)
        mask[:, : ny // 3] = 0
        case["mask"] = torch.from_numpy(mask).cuda()
    print("sampled sweeps", shape, block, fp, bp, masked, voxel, flush=True)
    v, norm = run(case)
    w, ref = run(case, flags=LDS)
    np.testing.assert_array_equal(v, w)
    assert norm == ref
    assert timed_kernel(case) == SWEEPING and timed_kernel(case, LDS) == FUSED
    r = A.BlockIterativeReconstructionOperator(**case)
    r.run_iterations(1)
    r.set_tile(*r.tile())
    r.run_iterations(1)
    np.testing.assert_array_equal(r.get_reconstructed_volume(dtype=torch.float32).cpu().numpy(), w)
