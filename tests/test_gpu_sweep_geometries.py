"""Separate sweeps (blocks, masks, oversampling) on detectors other than the
volume's own size and pitch, over z slabs and with 16-bit projections: the
fused passes' volume and residual norm bit for bit, and within the FP32 parity
bound (relative L2 1e-5; 2^-9 with 16-bit storage, as for the fused passes) of
the generic kernels.

Rows beside the volume and rows that share a plane, columns beside the volume,
detectors narrower than it, long-object compensation on rows without a plane;
one, two and four planes a workgroup with up to eight rays a thread: a forward
sweep of n projections takes four planes from 256 workgroups on (two with a
mask) and as many rays a thread, to eight, as leave 512 of them."""
import numpy as np
import pytest

import ettention_amd as E
from ettention_amd import api as A
from ettention_amd import synthetic as S

from _util import rel_l2

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SWEEPING = 3    # kernel of time_kernels
LDS, GENERIC = E.ETN_RECON_FLAG_LDS_BACK_PROJECTION, E.ETN_RECON_FLAG_GENERIC_KERNELS

# volume, detector, pitch, projections, block, options
CASES = {
    # rows beside the volume, with long-object compensation; four rows a plane and columns beside it
    "taller": ((132, 100, 168), (132, 160), (1.0, 1.0), 16, 8, dict(use_long_object_compensation=True)),
    "shorter": ((132, 100, 168), (132, 41), (1.0, 1.0), 16, 8, {}),
    "narrower": ((132, 100, 168), (70, 100), (1.0, 1.0), 16, 8, dict(use_long_object_compensation=True)),
    "wider": ((132, 100, 168), (250, 100), (1.0, 1.0), 16, 9, {}),
    "finer": ((132, 100, 168), (165, 400), (0.8, 0.25), 16, 8, {}),
    "coarser": ((134, 101, 160), (67, 101), (2.0, 1.0), 16, 8, {}),
    "slabs": ((132, 100, 168), (132, 110), (1.0, 1.0), 16, 8, dict(subvolumes=3)),
    "half_projections": ((132, 100, 200), (132, 110), (1.0, 1.0), 24, 8, dict(voxel_type="half", sixteen=True)),
    "bf16_projections": ((134, 101, 200), (134, 101), (1.0, 0.5), 24, 8, dict(voxel_type="bfloat16", sixteen=True)),
    # four planes a workgroup and 2, 4 and 8 rays a thread
    "two_rays": ((130, 1024, 130), (130, 1024), (1.0, 1.0), 8, 8, {}),
    "four_rays": ((140, 120, 136), (140, 2048), (1.0, 1.0), 8, 8, dict(use_long_object_compensation=True)),
    "eight_rays": ((302, 104, 72), (302, 2048), (1.0, 0.5), 8, 8, {}),
    "eight_rays_half": ((300, 104, 72), (300, 2048), (1.0, 1.0), 8, 8, dict(voxel_type="half")),
    # masks: one and two planes a workgroup, 2 and 4 rays a thread
    "mask_taller": ((92, 90, 70), (92, 130), (1.0, 1.0), 16, 8, dict(mask=True, use_long_object_compensation=True)),
    "mask_finer": ((92, 91, 70), (120, 182), (0.8, 0.5), 16, 8, dict(mask=True)),
    "mask_slabs": ((92, 90, 70), (92, 90), (1.0, 1.0), 16, 8, dict(mask=True, subvolumes=2)),
    "mask_two_rays": ((130, 64, 66), (130, 514), (1.0, 0.25), 8, 8, dict(mask=True, voxel_type="half")),
    "mask_four_rays": ((132, 64, 66), (132, 1030), (1.0, 1.0), 8, 8, dict(mask=True, voxel_type="bfloat16", sixteen=True)),
    # sub-rays and sample patterns
    "over_taller": ((104, 82, 100), (104, 120), (1.0, 1.0), 9, 1,
                    dict(fp_samples=2, bp_samples=4, use_long_object_compensation=True)),
    "over_wider": ((92, 82, 76), (140, 82), (1.0, 1.0), 9, 1, dict(fp_samples=3, bp_samples=9, mask=True)),
    "over_finer": ((92, 82, 76), (130, 164), (0.75, 0.5), 9, 2, dict(fp_samples=2, bp_samples=4)),
    "over_slabs": ((92, 82, 76), (92, 82), (1.0, 1.0), 9, 2, dict(bp_samples=9, subvolumes=2)),
    "over_eight_rays": ((104, 64, 84), (104, 2048), (1.0, 1.0), 8, 8, dict(fp_samples=4, bp_samples=4)),
    "over_mask_rays": ((102, 80, 84), (102, 1040), (1.0, 1.0), 8, 8, dict(fp_samples=4, bp_samples=4, mask=True)),
}


def reconstruct(case, flags):
    r = A.BlockIterativeReconstructionOperator(flags=flags, **case)
    r.run_iterations(2)
    return r.get_reconstructed_volume(dtype=torch.float32).cpu().numpy(), r.residual_norm()


@pytest.mark.parametrize("name", sorted(CASES))
def test_sweeps_on_other_detectors(name):
    size, det, pitch, count, block, opts = CASES[name]
    (nx, ny, nz), (nu, nv), (pu, pv) = size, det, pitch
    opts = dict(opts)
    base = E.ScannerGeometry.make((-0.5 * nu * pu, -0.5 * nv * pv, 500.0), (-0.5 * nu * pu, -0.5 * nv * pv, -500.0),
                                  (pu, 0, 0), (0, pv, 0), (nu, nv))
    tilts = np.linspace(-60.0, 60.0, count).astype(np.float32)
    whole = E.VolumeGeometry.make(size)
    phantom = S.ellipsoid_phantom((nz, ny, nx), seed=31, device=torch.device("cuda"))
    projections = torch.zeros((count, nv, nu), device="cuda")
    scratch = torch.zeros((nv, nu), device="cuda")
    for i, t in enumerate(tilts):
        A.forward_project(whole, phantom, A.rotate(base, float(t)), projections[i], scratch)
    if opts.pop("sixteen", False):
        projections = projections.to({"half": torch.float16, "bfloat16": torch.bfloat16}[opts["voxel_type"]])
    case = dict(volume=E.VolumeGeometry.make(size, subvolumes=opts.pop("subvolumes", 1)), base_geometry=base,
                tilt_angles=tilts, projections=projections, algorithm="blockiterative", block_size=block, lam=0.3,
                projection_iteration="identity")
    if opts.pop("mask", False):
        mask = np.random.default_rng(7).integers(0, 256, (nz, ny, nx)).astype(np.uint8)
        mask[:, : ny // 3] = 255
        case["mask"] = torch.from_numpy(mask).cuda()
    case.update(opts)
    print("sweep geometry", name, flush=True)
    kernel = A.BlockIterativeReconstructionOperator(**case).time_kernels()[0]
    assert kernel == SWEEPING
    v, norm = reconstruct(case, 0)
    w, ref = reconstruct(case, LDS)
    np.testing.assert_array_equal(v, w)
    assert norm == ref
    g, gnorm = reconstruct(dict(case, volume=whole), GENERIC)
    bound = 1e-5 if case.get("voxel_type", "float") == "float" else 2.0 ** -9
    assert rel_l2(v, g) <= bound
    assert abs(norm - gnorm) <= bound * gnorm
