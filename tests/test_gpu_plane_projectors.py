"""Single forward and back projections of single-axis tilts (one workgroup per
few detector rows, csrc/plane_projectors.hip) against the oracle: they perform
the oracle's float operations one for one, so the results are equal bit for bit."""
import numpy as np
import pytest

import ettention_amd as E
from ettention_amd import api as A
from oracle import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

TORCH = {"float": torch.float32, "half": torch.float16, "bfloat16": torch.bfloat16}

# (nx, ny, nz), detector (nu, nv), pitch, tilt: columns per thread 1, 2 and 4,
# one and two rows a workgroup (nv >= 512), rows without a plane and planes with
# several rows, nx off a multiple of 4, rays along x and z, volumes of one band
# and of a remainder, detectors narrower and wider than the volume
CASES = [
    ((64, 64, 64), (64, 64), (1.0, 1.0), 33.0),
    ((64, 5, 70), (64, 5), (1.0, 1.0), 0.0),
    ((64, 5, 70), (64, 5), (1.0, 1.0), 90.0),
    ((61, 7, 33), (61, 7), (1.0, 1.0), -47.5),
    ((40, 9, 50), (96, 30), (0.5, 0.5), 225.0),
    ((40, 9, 50), (20, 4), (2.0, 2.0), 12.0),
    ((516, 3, 41), (516, 3), (1.0, 1.0), 61.0),
    ((1030, 2, 37), (1030, 2), (1.0, 1.0), -30.0),
    ((96, 520, 24), (96, 520), (1.0, 1.0), 20.0),
    ((97, 513, 11), (97, 513), (1.0, 1.0), -75.0),
    ((700, 4, 300), (700, 4), (1.0, 1.0), 45.0),
]


def case(size, det, pitch, tilt, seed):
    nx, ny, nz = size
    vg, ov = E.VolumeGeometry.make(size), O.Volume.make(size)
    (nu, nv), (pu, pv) = det, pitch
    half = (-0.5 * nu * pu, -0.5 * nv * pv)
    base = ((half[0], half[1], float(nx)), (half[0], half[1], -float(nx)), (pu, 0, 0), (0, pv, 0), det)
    g = A.rotate(E.ScannerGeometry.make(*base), tilt)
    og = O.Scanner.make(g.source, g.detector, g.horizontal_pitch, g.vertical_pitch, g.resolution)
    return vg, ov, g, og, np.random.default_rng(seed)


@pytest.mark.parametrize("dtype", ["float", "half", "bfloat16"])
@pytest.mark.parametrize("size,det,pitch,tilt", CASES)
def test_forward_equals_the_oracle(size, det, pitch, tilt, dtype):
    vg, ov, g, og, rng = case(size, det, pitch, tilt, 3)
    vol = torch.from_numpy(rng.uniform(-1, 1, size[::-1]).astype(np.float32)).to(TORCH[dtype])
    start = rng.uniform(-1, 1, (2, det[1], det[0])).astype(np.float32)
    p, l = torch.from_numpy(start[0]).cuda(), torch.from_numpy(start[1]).cuda()
    A.forward_project(vg, vol.cuda(), g, p, l)
    op, ol = O.forward_project(ov, vol.float().numpy(), og, proj=start[0].copy(), length=start[1].copy())
    np.testing.assert_array_equal(p.cpu().numpy(), op)
    np.testing.assert_array_equal(l.cpu().numpy(), ol)


@pytest.mark.parametrize("dtype", ["float", "half", "bfloat16"])
@pytest.mark.parametrize("size,det,pitch,tilt", CASES)
def test_back_equals_the_oracle(size, det, pitch, tilt, dtype):
    vg, ov, g, og, rng = case(size, det, pitch, tilt, 4)
    vol = torch.from_numpy(rng.uniform(-1, 1, size[::-1]).astype(np.float32)).to(TORCH[dtype])
    residual = rng.normal(0, 1, det[::-1]).astype(np.float32)
    length = rng.uniform(0.5, 40, det[::-1]).astype(np.float32)
    length[:, : det[0] // 8] = 0.0            # rays beside the volume
    v = vol.cuda()
    A.back_project(vg, v, g, torch.from_numpy(residual).cuda(), torch.from_numpy(length).cuda(), lam=0.3, block_size=2)
    ref = vol.float().numpy().copy()
    O.back_project(ov, ref, og, residual, length, lam=0.3, block_size=2)
    ref = torch.from_numpy(ref).to(TORCH[dtype])   # the kernel rounds the updated voxel to storage once
    np.testing.assert_array_equal(v.float().cpu().numpy(), ref.float().numpy())


@pytest.mark.parametrize("subvolumes", [1, 3])
def test_slabs_add_up(subvolumes):
    vg, ov, g, og, rng = case((48, 6, 40), (48, 6), (1.0, 1.0), 25.0, 5)
    vg.subvolume_count = ov.slabs = subvolumes
    vol = rng.uniform(0, 1, (40, 6, 48)).astype(np.float32)
    p = torch.zeros((6, 48), device="cuda")
    l = torch.zeros_like(p)
    op, ol = np.zeros((6, 48), np.float32), np.zeros((6, 48), np.float32)
    for i in range(subvolumes):
        A.forward_project(vg, torch.from_numpy(vol).cuda(), g, p, l, subvolume=i)
        O.forward_project(ov, vol, og, slab=i, proj=op, length=ol)
    np.testing.assert_array_equal(p.cpu().numpy(), op)
    np.testing.assert_array_equal(l.cpu().numpy(), ol)


# rows whose rays run along a face of the volume (not this path's): the first and
# the last one, ones in between, one of a coarser detector, none
@pytest.mark.parametrize("nv,pitch", [(7, 1.0), (9, 1.0), (4, 2.0), (13, 0.5), (8, 1.0)])
def test_rows_on_a_face_equal_the_oracle(nv, pitch):
    size = (48, 6, 40)
    vg, ov, g, og, rng = case(size, (48, nv), (1.0, pitch), 25.0, 6)
    vol = rng.uniform(0, 1, size[::-1]).astype(np.float32)
    p = torch.zeros((nv, 48), device="cuda")
    l = torch.zeros_like(p)
    A.forward_project(vg, torch.from_numpy(vol).cuda(), g, p, l)
    op, ol = O.forward_project(ov, vol, og)
    np.testing.assert_array_equal(p.cpu().numpy(), op)
    np.testing.assert_array_equal(l.cpu().numpy(), ol)


# workgroups of 256, 128 and 64 columns (one, two and four rows of waves for the
# slices), one column more than those, fewer slices than waves
@pytest.mark.parametrize("nx", [64, 65, 128, 129, 192, 193, 256, 257, 260, 320, 321])
@pytest.mark.parametrize("nz,tilt,dtype", [(3, 10.0, "float"), (37, 60.0, "bfloat16"), (130, -35.0, "half")])
def test_back_of_every_row_width_equals_the_oracle(nx, nz, tilt, dtype):
    test_back_equals_the_oracle((nx, 5, nz), (nx, 5), (1.0, 1.0), tilt, dtype)
