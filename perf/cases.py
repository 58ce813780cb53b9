"""The framework's work as its users call it, for measuring how fast it is.

Every case goes through the Python front end (`ettention_amd.api`,
`ettention_amd.learned`), the binding of the C ABI: the projection operators
one call at a time, whole reconstructions (SART, blocks, SIRT, weighted back
projection) and the learned correction (prediction and training gradient).

`listed()` names the cases, `draw(rng)` gives more of the same ranges,
`prepare(case, seed)` makes what a program holds before the call, `run(state)`
is one pass, `work(case)` the bytes and operations a pass cannot do without,
`exact(case, seed)` the pass's results in 64-bit torch arithmetic.
"""
import math
import os

import numpy as np
import torch

import ettention_amd as E
from ettention_amd import api as A
from ettention_amd import learned as Lrn
from ettention_amd import synthetic as S

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NET_PARAMS = os.path.join(ROOT, "ettention_amd", "data", "correction_net_512.npy")

DTYPES = {"float": torch.float32, "half": torch.float16, "bfloat16": torch.bfloat16}
LAMBDA = 0.3
EPSILON = 1e-4           # rays and ray lengths below this count as a miss
MAX_STEPS = 2048         # voxels a ray visits at most


def _projector(kind, name, size, dtype, tilt, xtilt=0.0, samples=1, mask=False):
    nx, ny, nz = size
    return {"name": name, "kind": kind, "nx": nx, "ny": ny, "nz": nz, "dtype": dtype, "tilt": tilt, "xtilt": xtilt,
            "samples": samples, "mask": mask}


def _reconstruction(name, size, tilts, dtype="float", block=1, order="random", iterations=1, fp_samples=1,
                    bp_samples=1, mask=False, xtilt=0.0):
    nx, ny, nz = size
    return {"name": name, "kind": "reconstruct", "nx": nx, "ny": ny, "nz": nz, "tilts": tilts, "dtype": dtype,
            "block": block, "order": order, "iterations": iterations, "fp_samples": fp_samples,
            "bp_samples": bp_samples, "mask": mask, "xtilt": xtilt}


def listed():
    return [
        # one operator call on a small volume, as a host program that drives
        # its own loop over test data makes it: launches and host work count
        _projector("forward", "forward_64", (64, 64, 64), "float", 33.0),
        # one operator call on the volume of the throughput benchmark
        _projector("forward", "forward_512", (512, 512, 512), "float", 33.0),
        _projector("back", "back_512", (512, 512, 512), "float", 33.0),
        # the operators with everything on: odd sizes, 16-bit storage, a mask
        # of known support, oversampling, a tilt axis that is not quite y
        _projector("forward", "forward_odd_f16", (301, 203, 257), "half", -47.0, xtilt=4.0, samples=2, mask=True),
        _projector("back", "back_odd_bf16", (301, 203, 257), "bfloat16", -47.0, xtilt=4.0, samples=4, mask=True),
        # a small tilt series reconstructed start to finish (10 iterations in
        # acquisition order)
        _reconstruction("sart_128", (128, 128, 64), 61, order="identity", iterations=10),
        # one iteration of the throughput benchmark
        _reconstruction("sart_512", (512, 512, 512), 121),
        # blocks of eight projections in random order on a thick slab
        _reconstruction("block8_512", (512, 512, 256), 121, block=8),
        # the oversampled, masked reconstruction of the reference's sample
        # parameter files (4 x 4 sub-rays, 9 samples a voxel) on an odd-sized
        # bf16 volume
        _reconstruction("sart_over_bf16", (250, 300, 150), 61, dtype="bfloat16", fp_samples=4, bp_samples=9,
                        mask=True),
        # weighted back projection of a whole series: the quick look at it
        {"name": "wbp_512", "kind": "wbp", "nx": 512, "ny": 512, "nz": 512, "tilts": 121},
        # the learned correction of an early iterate, and one training gradient
        # on the crop size that training takes
        {"name": "predict_256", "kind": "predict", "nx": 256, "ny": 256, "nz": 256},
        {"name": "gradient_128", "kind": "gradient", "nx": 128, "ny": 128, "nz": 128},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward", "back", "reconstruct", "reconstruct", "wbp", "predict", "gradient"])
    if kind in ("predict", "gradient"):
        # the network halves its volume twice: multiples of 4
        hi = 256 if kind == "predict" else 128
        n = [4 * _log_int(rng, 4, hi // 4) for _ in range(3)]
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2]}
    n = [_log_int(rng, 48, 512) for _ in range(3)]
    if kind == "wbp":
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "tilts": rng.randint(21, 121)}
    dtype = rng.choice(["float", "float", "half", "bfloat16"])
    mask = rng.random() < 0.3
    xtilt = rng.choice([0.0, 0.0, round(rng.uniform(-8.0, 8.0), 2)])
    if kind in ("forward", "back"):
        c = _projector(kind, None, n, dtype, round(rng.uniform(-75.0, 75.0), 2), xtilt,
                       rng.choice([1, 1, 2] if kind == "forward" else [1, 1, 4]), mask)
    else:
        over = rng.random() < 0.25
        c = _reconstruction(None, n, rng.randint(21, 121), dtype, rng.choice([1, 1, 4, 8, 0]),
                            rng.choice(["random", "identity"]), 1, rng.choice([2, 4]) if over else 1,
                            rng.choice([4, 9]) if over else 1, mask, xtilt)
        # no more work than the largest listed case: the oversampled and the
        # two-axis geometries cost many times a plain one
        cost = (10 if over else 1) * (12 if xtilt else 1)
        while c["nx"] * c["ny"] * c["nz"] * c["tilts"] * cost > 512 ** 3 * 121:
            for k in ("nx", "ny", "nz"):
                c[k] = max(32, int(c[k] * 0.8))
    del c["name"]
    return c


# ---- inputs ----------------------------------------------------------------

def _angles(n):
    return np.linspace(-60.0, 60.0, n).astype(np.float32)


def _rotation(tilt, xtilt):
    """Columns of the scanner's rotation in float64: -tilt about the y axis,
    and with an x-axis tilt first the points, then the axis, turned about x."""
    t, a = -math.radians(tilt), math.radians(xtilt)
    c, s = math.cos(t), math.sin(t)
    if xtilt == 0.0:
        return np.array([[c, 0.0, -s], [0.0, 1.0, 0.0], [s, 0.0, c]])
    ca, sa = math.cos(a), math.sin(a)
    about_x = np.array([[1.0, 0.0, 0.0], [0.0, ca, sa], [0.0, -sa, ca]])
    ay, az = ca, -sa                       # the tilt axis
    o = 1.0 - c
    about_axis = np.array([[c, -s * az, s * ay], [s * az, c + o * ay * ay, o * ay * az],
                           [-s * ay, o * ay * az, c + o * az * az]])
    return about_axis @ about_x


def _geometry(nx, ny, tilt, xtilt):
    """source, horizontal pitch, vertical pitch and ray direction of a tilted
    scanner with an nx x ny detector, in float64."""
    r = _rotation(float(tilt), float(xtilt))
    source = r @ np.array([-0.5 * nx, -0.5 * ny, float(nx)])
    return source, r @ [1.0, 0.0, 0.0], r @ [0.0, 1.0, 0.0], r @ [0.0, 0.0, -1.0]


def _phantom(case, seed):
    return S.ellipsoid_phantom((case["nz"], case["ny"], case["nx"]), seed=1000 + seed, device="cuda")


def _projections(case, angles, xtilt, seed):
    """The phantom's tilt series in closed form (chords of its ellipsoids),
    with 2 % Gaussian noise: no projector of this package makes the inputs."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    ells, _ = S.phantom_parameters((nz, ny, nx), 1000 + seed)
    centre = 0.5 * np.array([nx, ny, nz], np.float64)
    geos = [_geometry(nx, ny, a, xtilt) for a in angles]
    u = torch.arange(nx, dtype=torch.float64, device="cuda") + 0.5
    v = torch.arange(ny, dtype=torch.float64, device="cuda") + 0.5
    out = torch.zeros((len(angles), ny, nx), dtype=torch.float32, device="cuda")
    for i, (src, h, w, ray) in enumerate(geos):
        total = torch.zeros((ny, nx), dtype=torch.float64, device="cuda")
        for c, ax, rot, density in ells:
            turn = (rot / ax).T             # world offsets to the unit sphere
            o, du, dv, d = (turn @ (src - (c - centre)), turn @ h, turn @ w, turn @ ray)
            dd = float(d @ d)
            # |o + u du + v dv + t d| = 1: discriminant in u and v
            od = float(o @ d) + u[None, :] * float(du @ d) + v[:, None] * float(dv @ d)
            oo = (float(o @ o) + u[None, :] * (2.0 * float(o @ du)) + v[:, None] * (2.0 * float(o @ dv)) +
                  u[None, :] ** 2 * float(du @ du) + v[:, None] ** 2 * float(dv @ dv) +
                  (2.0 * float(du @ dv)) * u[None, :] * v[:, None])
            disc = od * od - dd * (oo - 1.0)
            total += disc.clamp_(min=0.0).sqrt_() * (2.0 * density / dd)
        out[i] = total
    g = torch.Generator(device="cuda").manual_seed(seed)
    sigma = 0.02 * float(out.max())
    return out + sigma * torch.randn(out.shape, generator=g, device="cuda")


def _mask(case):
    """255 inside a y-axis cylinder that holds the specimen, fading to 0."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    x = torch.arange(nx, device="cuda") + 0.5 - 0.5 * nx
    z = torch.arange(nz, device="cuda") + 0.5 - 0.5 * nz
    r = (x[None, :] ** 2 + z[:, None] ** 2).sqrt() / (0.45 * nx)
    m = ((1.1 - r) * 2550.0).clamp(0.0, 255.0).to(torch.uint8)
    return m[:, None, :].expand(nz, ny, nx).contiguous()


def _images(case, seed):
    """A residual image (structured, both signs) and the ray lengths that go with it."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    residual = torch.randn((ny, nx), generator=g, device="cuda") * (0.02 * nz)
    lengths = float(nz) * (1.0 + 0.05 * torch.rand((ny, nx), generator=g, device="cuda"))
    edge = torch.arange(nx, device="cuda")
    lengths[:, (edge < nx // 16) | (edge >= nx - nx // 16)] = 0.0      # rays beside the volume
    return residual, lengths


def _iterate(case, seed):
    """An early iterate (the phantom blurred along the missing wedge, with
    noise), its last update, and the late iterate it should become."""
    late = _phantom(case, seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    k = 3
    x = torch.nn.functional.avg_pool3d(late[None, None], (2 * k + 1, 1, 1), 1, (k, 0, 0))[0, 0].contiguous()
    x = x + 0.05 * torch.randn(x.shape, generator=g, device="cuda")
    d = 0.1 * (late - x) + 0.01 * torch.randn(x.shape, generator=g, device="cuda")
    return x, d.contiguous(), late


NET_SCALE = 1.0


def prepare(case, seed):
    kind = case["kind"]
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if kind in ("predict", "gradient"):
        x, d, late = _iterate(case, seed)
        net = Lrn.CorrectionNet((nz, ny, nx), np.load(NET_PARAMS))
        return {"kind": kind, "net": net, "x": x, "d": d, "late": late, "out": torch.empty_like(x)}
    vg = E.VolumeGeometry.make((nx, ny, nz))
    base = E.ScannerGeometry.mrc_base(nx, ny)
    if kind in ("forward", "back"):
        s = {"kind": kind, "vg": vg, "g": A.rotate(base, case["tilt"], case["xtilt"]), "samples": case["samples"],
             "volume": _phantom(case, seed).to(DTYPES[case["dtype"]]),
             "mask": _mask(case) if case["mask"] else None}
        if kind == "forward":
            s["p"] = torch.zeros((ny, nx), dtype=torch.float32, device="cuda")
            s["l"] = torch.zeros_like(s["p"])
        else:
            s["residual"], s["lengths"] = _images(case, seed)
        return s
    angles = _angles(case["tilts"])
    xtilt = case.get("xtilt", 0.0)
    projections = _projections(case, angles, xtilt, seed)
    common = dict(volume=vg, base_geometry=base, tilt_angles=angles, projections=projections)
    if kind == "wbp":
        op = A.WeightedBackProjection(lam=1.0, **common)
        dtype, iterations = torch.float32, None
    else:
        block = case["block"]
        op = A.BlockIterativeReconstructionOperator(
            algorithm="sart" if block == 1 else "sirt" if block == 0 else "blockiterative", block_size=block,
            lam=LAMBDA, fp_samples=case["fp_samples"], bp_samples=case["bp_samples"],
            projection_iteration=case["order"], voxel_type=case["dtype"], x_axis_tilt=xtilt,
            mask=_mask(case) if case["mask"] else None, **common)
        dtype, iterations = DTYPES[case["dtype"]], case["iterations"]
    return {"kind": kind, "op": op, "start": torch.zeros((nz, ny, nx), dtype=dtype, device="cuda"),
            "iterations": iterations}


# ---- one pass ----------------------------------------------------------------

def run(s):
    kind = s["kind"]
    if kind == "forward":
        s["p"].zero_()
        s["l"].zero_()
        A.forward_project(s["vg"], s["volume"], s["g"], s["p"], s["l"], samples=s["samples"], mask=s["mask"])
        return s["p"], s["l"]
    if kind == "back":
        A.back_project(s["vg"], s["volume"], s["g"], s["residual"], s["lengths"], lam=LAMBDA, samples=s["samples"],
                       mask=s["mask"])
        return s["volume"]
    if kind == "predict":
        return s["net"].predict(s["x"], s["d"], NET_SCALE, out=s["out"])
    if kind == "gradient":
        loss, g = s["net"].gradient(s["x"], s["d"], s["late"], NET_SCALE)
        return loss, g
    op = s["op"]
    op.set_volume(s["start"])
    if kind == "wbp":
        op.run()
    else:
        op.run_iterations(s["iterations"])
    return op.get_reconstructed_volume()


# ---- what a pass cannot do without ------------------------------------------

def work(case):
    kind = case["kind"]
    V, P = case["nx"] * case["ny"] * case["nz"], case["nx"] * case["ny"]
    if kind in ("predict", "gradient"):
        f = sum(2.0 * 27.0 * ci * co * (V / 8 ** {"1": 0, "2": 1, "3": 2, "4": 1, "5": 0}[name[1]])
                for name, ci, co in Lrn.LAYERS) + 32.0 * V
        # the backward pass costs the forward's twice, but for the input's own gradient
        return {"bytes": 12.0 * V, "flops": f if kind == "predict" else 3.0 * f - 2.0 * 27.0 * 2 * 16 * V}
    s = 4 if case.get("dtype", "float") == "float" else 2
    if kind == "forward":
        return {"bytes": (s + (1 if case["mask"] else 0)) * V + 16 * P, "flops": 4.0 * V * case["samples"] ** 2}
    if kind == "back":
        return {"bytes": (2 * s + (1 if case["mask"] else 0)) * V + 8 * P, "flops": 16.0 * V * case["samples"]}
    n = case["tilts"]
    if kind == "wbp":
        # the projections in, the volume read and written once
        return {"bytes": 2 * s * V + 4.0 * n * P, "flops": 16.0 * V * n + 256.0 * n * P}
    blocks = 1 if case["block"] == 0 else -(-n // case["block"])
    per = 4.0 * case["fp_samples"] ** 2 + 16.0 * case["bp_samples"]
    # a block's residuals need the whole volume, its update changes it: one read and one write a block
    return {"bytes": case["iterations"] * ((2 * s + (1 if case["mask"] else 0)) * V * blocks + 4.0 * n * P),
            "flops": case["iterations"] * per * V * n}


# ---- the same in 64 bits -----------------------------------------------------

def _ray_setup(size, src, ray):
    """Entry voxel, distances to the first borders and steps of rays through
    the box centred on 0 with unit voxels; borders lie on multiples of the
    voxel size in world coordinates."""
    res = torch.tensor(size, dtype=torch.float64, device="cuda")
    ray = torch.as_tensor(ray, dtype=torch.float64, device="cuda").expand_as(src)
    ray = torch.where(ray.abs() < 1e-15, torch.zeros_like(ray), ray)
    still = ray == 0.0
    inv = torch.where(still, torch.full_like(ray, -1e300), 1.0 / ray)
    lo, hi = -0.5 * res, 0.5 * res
    t0, t1 = (lo - src) * inv, (hi - src) * inv
    t_in = torch.minimum(t0, t1).amax(-1)
    t_out = torch.maximum(t0, t1).amin(-1)
    live = t_out - t_in > EPSILON
    p = torch.minimum(torch.maximum(src + t_in[:, None] * ray, lo), hi)
    vox = torch.minimum((p - lo).floor(), res - 1).clamp_(min=0.0).long()
    border = p.floor()
    first = torch.where(ray > 0.0, (border + 1.0 - p) * inv, (border - p) * inv)
    step = inv.abs()
    first = torch.where(first == 0.0, step, first)
    first = torch.where(still, torch.full_like(first, 1e300), first)
    return vox, first, step, torch.sign(ray).long(), live


def _trace(size, src, ray, visit):
    """Walks the rays voxel by voxel; visit(linear voxel index, segment length)."""
    nx, ny, nz = size
    vox, rest, step, sign, live = _ray_setup(size, src, ray)
    res = torch.tensor(size, device="cuda")
    for k in range(MAX_STEPS):
        live = live & ((vox >= 0) & (vox < res)).all(-1)
        if k % 32 == 0 and not bool(live.any()):
            break
        dt, axis = rest.min(-1)
        at = torch.where(live, (vox[:, 2] * ny + vox[:, 1]) * nx + vox[:, 0], torch.zeros_like(axis))
        visit(at, torch.where(live, dt, torch.zeros_like(dt)))
        taken = torch.nn.functional.one_hot(axis, 3).bool()
        rest = torch.where(taken, step, rest - dt[:, None])
        vox = vox + taken * sign


def _exact_forward(case, seed):
    nx, ny, nz = size = case["nx"], case["ny"], case["nz"]
    volume = _phantom(case, seed).to(DTYPES[case["dtype"]]).double().reshape(-1)
    weight = _mask(case).double().reshape(-1) / 255.0 if case["mask"] else None
    src, h, v, ray = (torch.tensor(a, dtype=torch.float64, device="cuda")
                      for a in _geometry(nx, ny, np.float32(case["tilt"]), np.float32(case["xtilt"])))
    n = case["samples"]
    u = torch.arange(nx, dtype=torch.float64, device="cuda")
    w = torch.arange(ny, dtype=torch.float64, device="cuda")
    total, length = (torch.zeros(ny * nx, dtype=torch.float64, device="cuda") for _ in range(2))

    def visit(at, dt):
        total.add_(dt * volume[at])
        length.add_(dt if weight is None else dt * weight[at])

    for i in range(n):
        for j in range(n):
            origin = (src + h * (u + (0.5 + i) / n)[None, :, None] + v * (w + (0.5 + j) / n)[:, None, None])
            _trace(size, origin.reshape(-1, 3), ray, visit)
    return (total / n ** 2).reshape(ny, nx), (length / n ** 2).reshape(ny, nx)


def _pattern(h, v, ray, samples):
    """Sample offsets inside a unit voxel, on the detector's axes, and the
    chord of the ray through each."""
    m = int(round(math.sqrt(samples)))
    out = []
    for y in range(m):
        for x in range(m):
            p = ((x + 0.5) / m - 0.5) * h + ((y + 0.5) / m - 0.5) * v
            t = [sorted(((-0.5 - p[k]) / ray[k], (0.5 - p[k]) / ray[k])) for k in range(3) if abs(ray[k]) > 1e-15]
            out.append((p, min(b for _, b in t) - max(a for a, _ in t)))
    return out


def _lookup(image, u, v):
    """Bilinear, zero outside the image; (u, v) with pixel centres on integers."""
    ny, nx = image.shape
    padded = torch.nn.functional.pad(image, (2, 2, 2, 2))
    fu, fv = u.floor(), v.floor()
    tu, tv = u - fu, v - fv
    i = fu.clamp(-2, nx).long() + 2
    j = fv.clamp(-2, ny).long() + 2
    flat, wide = padded.reshape(-1), nx + 4
    at = j * wide + i
    i1 = (i + 1).clamp(max=nx + 3) - i
    j1 = ((j + 1).clamp(max=ny + 3) - j) * wide
    a = flat[at] + (flat[at + i1] - flat[at]) * tu
    b = flat[at + j1] + (flat[at + j1 + i1] - flat[at + j1]) * tu
    return a + (b - a) * tv


def _exact_back(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    volume = _phantom(case, seed).to(DTYPES[case["dtype"]]).double()
    weight = _mask(case).double() / 255.0 if case["mask"] else None
    residual, lengths = (t.double() for t in _images(case, seed))
    _, h, v, ray = _geometry(nx, ny, np.float32(case["tilt"]), np.float32(case["xtilt"]))
    x = torch.arange(nx, dtype=torch.float64, device="cuda") + 0.5 - 0.5 * nx
    y = torch.arange(ny, dtype=torch.float64, device="cuda") + 0.5 - 0.5 * ny
    for z in range(nz):
        pz = z + 0.5 - 0.5 * nz
        total = torch.zeros((ny, nx), dtype=torch.float64, device="cuda")
        used = torch.zeros_like(total)
        for p, chord in _pattern(h, v, ray, case["samples"]):
            u = (x + p[0])[None, :] * h[0] + (y + p[1])[:, None] * h[1] + (pz + p[2]) * h[2] + 0.5 * nx
            w = (x + p[0])[None, :] * v[0] + (y + p[1])[:, None] * v[1] + (pz + p[2]) * v[2] + 0.5 * ny
            L, R = _lookup(lengths, u, w), _lookup(residual, u, w)
            ok = L > EPSILON
            total += torch.where(ok, R * LAMBDA * chord / torch.where(ok, L, torch.ones_like(L)), torch.zeros_like(L))
            used += ok
        total = total / used.clamp(min=1.0)
        volume[z] += total if weight is None else total * weight[z]
    return volume


class _PlaneSeries:
    """Single-axis tilt, one sample: every ray stays in its plane y, and the
    volume is kept as [z * nx + x][y]."""

    def __init__(self, case, angles):
        self.nx, self.ny, self.nz = nx, ny, nz = case["nx"], case["ny"], case["nz"]
        self.geo = [_geometry(nx, ny, a, 0.0) for a in angles]
        u = torch.arange(nx, dtype=torch.float64, device="cuda") + 0.5
        src = torch.cat([torch.tensor(s, device="cuda") + torch.tensor(h, device="cuda") * u[:, None]
                         for s, h, _, _ in self.geo])
        src[:, 1] = 0.0
        ray = torch.cat([torch.tensor(r, device="cuda").expand(nx, 3) for *_, r in self.geo])
        self.at, self.dt = [], []
        _trace((nx, 1, nz), src, ray, lambda at, dt: (self.at.append(at.int()), self.dt.append(dt)))
        self.at, self.dt = torch.stack(self.at), torch.stack(self.dt)
        self.x = torch.arange(nx, dtype=torch.float64, device="cuda") + 0.5 - 0.5 * nx
        self.z = torch.arange(nz, dtype=torch.float64, device="cuda") + 0.5 - 0.5 * nz

    def forward(self, volume, i):
        """([ny][nx] line integrals, [ny][nx] lengths) of projection i."""
        nx = self.nx
        at, dt = self.at[:, i * nx:(i + 1) * nx], self.dt[:, i * nx:(i + 1) * nx]
        out = torch.zeros((nx, self.ny), dtype=torch.float64, device="cuda")
        for k in range(0, at.shape[0], 128):
            part = at[k:k + 128].long()
            out += (volume[part.reshape(-1)].reshape(*part.shape, -1) * dt[k:k + 128, :, None]).sum(0)
        return out.T, dt.sum(0).expand(self.ny, nx)

    def back(self, volume, i, residual, lengths, lam):
        """volume += lam R chord / L for every voxel; images [ny][nx]."""
        _, h, v, ray = self.geo[i]
        chord = _pattern(h, v, ray, 1)[0][1]
        # detector rows y and y + 1 count one half each in plane y
        rows = [(0.5 * (m + torch.cat([m[1:], torch.zeros_like(m[:1])]))).T.contiguous() for m in (residual, lengths)]
        rows = [torch.nn.functional.pad(m, (0, 0, 2, 3)) for m in rows]
        step = max(1, (1 << 25) // (self.nx * self.ny))
        for z0 in range(0, self.nz, step):
            z = self.z[z0:z0 + step]
            u = (self.x[None, :] * h[0] + z[:, None] * h[2]).reshape(-1) + 0.5 * self.nx
            f = u.floor()
            t = (u - f)[:, None]
            k = f.clamp(-2, self.nx).long() + 2
            R, L = (m[k] + (m[k + 1] - m[k]) * t for m in rows)
            ok = L > EPSILON
            volume[z0 * self.nx:(z0 + len(z)) * self.nx] += torch.where(
                ok, R * (lam * chord) / torch.where(ok, L, torch.ones_like(L)), torch.zeros_like(L))

    def result(self, volume):
        return volume.reshape(self.nz, self.nx, self.ny).transpose(1, 2).contiguous()


def _exact_reconstruct(case, seed):
    n, V = case["tilts"], case["nx"] * case["ny"] * case["nz"]
    # (the random order is the reference generator's own; the oversampled and two-axis ones take too long)
    if (case["order"] != "identity" or case["fp_samples"] * case["bp_samples"] != 1 or case["mask"] or case["xtilt"]
            or V * n * case["iterations"] > 512 ** 3 * 121):
        return None
    angles = _angles(n)
    projections = _projections(case, angles, 0.0, seed).double()
    series = _PlaneSeries(case, angles)
    volume = torch.zeros((case["nz"] * case["nx"], case["ny"]), dtype=torch.float64, device="cuda")
    size = n if case["block"] == 0 else case["block"]
    for _ in range(case["iterations"]):
        for b in range(0, n, size):
            block = range(b, min(n, b + size))
            images = []
            for i in block:
                p, length = series.forward(volume, i)
                images.append((projections[i] - p, length))
            for i, (r, length) in zip(block, images):
                series.back(volume, i, r, length, LAMBDA / len(block))
    return series.result(volume)


def _mirror(n, size):
    """Source index of each column of a row padded to `size` by mirroring."""
    x = np.arange(size)
    lo, hi = (size - n) // 2, (size + n) // 2
    m = np.where((x >= lo) & (x < hi), x - lo, np.where(x < hi, lo - x, n + hi - 1 - x))
    return torch.from_numpy(np.clip(m, 0, n - 1)).cuda()


def _exact_wbp(case, seed):
    nx, ny, n = case["nx"], case["ny"], case["tilts"]
    angles = _angles(n)
    projections = _projections(case, angles, 0.0, seed).double()
    taps = 128
    ux, uy = (1 << (max(k, 1) - 1).bit_length() for k in (max(taps, nx), ny))
    padded = projections[:, _mirror(ny, uy)][:, :, _mirror(nx, ux)]
    padded = torch.roll(padded, -1, 1)[:, uy // 2 - ny // 2:uy // 2 - ny // 2 + ny]
    filtered = torch.zeros_like(padded)
    for t in range(taps):
        p = t - taps // 2
        if p == 0:
            filtered += 0.25 * padded
        elif p % 2:
            filtered -= torch.roll(padded, p, 2) / (math.pi ** 2 * p * p)
    filtered = filtered[:, :, ux // 2 - nx // 2:ux // 2 - nx // 2 + nx]
    series = _PlaneSeries(case, angles)
    volume = torch.zeros((case["nz"] * nx, ny), dtype=torch.float64, device="cuda")
    u = torch.arange(nx, dtype=torch.float64, device="cuda") + 0.5
    for i, (src, h, _, ray) in enumerate(series.geo):
        t = []
        for k, size in ((0, nx), (2, case["nz"])):
            if abs(ray[k]) > 1e-15:
                o = src[k] + u * h[k]
                a, b = (-0.5 * size - o) / ray[k], (0.5 * size - o) / ray[k]
                t.append((torch.minimum(a, b), torch.maximum(a, b)))
        t_in = torch.stack([a for a, _ in t]).amax(0)
        t_out = torch.stack([b for _, b in t]).amin(0)
        series.back(volume, i, filtered[i], (t_out - t_in).clamp(min=0.0).expand(ny, nx), 1.0 / n)
    return series.result(volume)


def _net_parameters():
    flat = torch.from_numpy(np.load(NET_PARAMS)).cuda().double().requires_grad_()
    out, at = [], 0
    for _, ci, co in Lrn.LAYERS:
        w = flat[at:at + co * 27 * ci].reshape(co, 27, ci)
        at += co * 27 * ci
        out.append((w, flat[at:at + co]))
        at += co
    return flat, out, flat[at:at + 16], flat[at + 16]


def _net_forward(layers, head, bias, x, d):
    """The correction network in float64, channels last."""
    def conv(a, k):
        w, b = layers[k]
        D, H, W, ci = a.shape
        p = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1, 1, 1))
        y = b.expand(D * H * W, -1)
        for t in range(27):
            z0, y0, x0 = t // 9, t // 3 % 3, t % 3
            y = y + p[z0:z0 + D, y0:y0 + H, x0:x0 + W].reshape(-1, ci) @ w[:, t].T
        return torch.relu(y).reshape(D, H, W, -1)

    def pool(a):
        D, H, W, c = a.shape
        return a.reshape(D // 2, 2, H // 2, 2, W // 2, 2, c).mean((1, 3, 5))

    def up(a):
        return a.repeat_interleave(2, 0).repeat_interleave(2, 1).repeat_interleave(2, 2)

    one = conv(conv(torch.stack([x, d], -1), 0), 1)
    two = conv(conv(pool(one), 2), 3)
    three = conv(conv(pool(two), 4), 5)
    four = conv(conv(torch.cat([up(three), two], -1), 6), 7)
    five = conv(conv(torch.cat([up(four), one], -1), 8), 9)
    return x + (five * head).sum(-1) + bias


def _exact_network(case, seed):
    x, d, late = (t.double() for t in _iterate(case, seed))
    flat, layers, head, bias = _net_parameters()
    xs, ds = x * NET_SCALE, d * (NET_SCALE * Lrn.UPDATE_GAIN)
    if case["kind"] == "predict":
        with torch.no_grad():
            return _net_forward(layers, head, bias, xs, ds) / NET_SCALE
    loss = ((_net_forward(layers, head, bias, xs, ds) - late * NET_SCALE) ** 2).mean()
    loss.backward()
    return float(loss.detach()), flat.grad


def exact(case, seed):
    kind = case["kind"]
    if kind == "forward":
        return _exact_forward(case, seed)
    if kind == "back":
        return _exact_back(case, seed)
    if kind == "wbp":
        return _exact_wbp(case, seed)
    if kind == "reconstruct":
        return _exact_reconstruct(case, seed)
    return _exact_network(case, seed)
