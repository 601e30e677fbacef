"""Workloads of the X-ray projectors: the work that a reconstruction program has the library do.

A case is a dict of plain values:
  kind    "project"  one forward and / or back projection through a projector's apply / applyAdjoint
          "cgls"     a whole CGLS solve on one projector
          "batch"    a whole FISTA solve (L1) on a batch of uneven 2D problems, in hipGraphs
          "step"     a training step through the differentiable projector: loss, backward, update
  method  joseph, siddon, blob, bspline, pcblob, pcbspline (the last two: phase contrast)
  dtype   f32, f64, bf16: the storage type of volume and sinogram
  way     forward, adjoint or both (kind "project")
  vol     voxels as "x,y[,z]"; det: detector pixels as "u[,v]"; poses: of a full circle
  arc     detector angle in radians of a curved detector, 0 for a planar one

listed() gives the fixed cases, draw(rng) one more of the same ranges, prepare(case, seed) what
a program has in hand before the call, run(state) one pass, work(case) the bytes and operations
a pass cannot do without, exact(case, seed) the same outputs in 64-bit arithmetic by plain torch.
"""
import math

import numpy as np
import torch

import elsa_amd as E
from elsa_amd.autograd import project

CLASSES = {"joseph": E.JosephsMethodCUDA, "siddon": E.SiddonsMethodCUDA, "blob": E.BlobVoxelProjectorCUDA,
           "bspline": E.BSplineVoxelProjectorCUDA, "pcblob": E.PhaseContrastBlobVoxelProjectorCUDA,
           "pcbspline": E.PhaseContrastBSplineVoxelProjectorCUDA}
DTYPES = {"f32": np.float32, "f64": np.float64, "bf16": "bfloat16"}
TORCH = {"f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16}
SUPPORT = {"blob": 2.0, "pcblob": 2.0, "bspline": 1.5, "pcbspline": 1.5}  # footprint radius in voxels
MAGNIFICATION = 1.05  # source-centre 100 N, centre-detector 5 N
LAMBDA_TV, STEP, LAMBDA_L1 = 0.01, 1.0e-5, 1.0e-3


def _case(name, kind, method, dtype, way, vol, det, poses, arc=0.0, problems=0, iterations=0, volumes=0):
    return {"name": name, "kind": kind, "method": method, "dtype": dtype, "way": way, "vol": vol, "det": det,
            "poses": poses, "arc": arc, "problems": problems, "iterations": iterations, "volumes": volumes}


def listed():
    return [
        # the smallest call: one slice of a 2D test problem, where launches and latency count
        _case("joseph2d_64", "project", "joseph", "f32", "both", "64,64", "91", 90),
        # the 2D fan-beam benchmark size: one slice of a scan inside an iterative method
        _case("joseph2d_256", "project", "joseph", "f32", "both", "256,256", "384", 180),
        # elsa's data_t = double operators on a small odd volume (no axis a multiple of a tile)
        _case("joseph3d_ragged_f64", "project", "joseph", "f64", "both", "97,61,113", "167,95", 77),
        # the headline cone-beam scan, forward and back
        _case("joseph3d_256_forward", "project", "joseph", "f32", "forward", "256,256,256", "384,384", 360),
        _case("joseph3d_256_adjoint", "project", "joseph", "f32", "adjoint", "256,256,256", "384,384", 360),
        # the largest: a 512^3 scan held in bfloat16
        _case("joseph3d_512_bf16", "project", "joseph", "bf16", "both", "512,512,512", "768,768", 720),
        # the same scan as the headline with exact intersection lengths
        _case("siddon3d_256", "project", "siddon", "f32", "both", "256,256,256", "384,384", 360),
        # smooth basis functions: an odd-sized blob scan in FP32, a B-spline one in FP64
        _case("blob3d_ragged", "project", "blob", "f32", "both", "131,125,119", "193,187", 180),
        _case("bspline3d_96_f64", "project", "bspline", "f64", "both", "96,96,96", "144,144", 90),
        # whole reconstructions: 64 uneven 2D problems at once in hipGraphs, and one 3D scan
        _case("fista_batch2d_64", "batch", "joseph", "f32", "both", "128,512", "0", 360, problems=64, iterations=20),
        _case("cgls3d_128", "cgls", "joseph", "f32", "both", "128,128,128", "192,192", 180, iterations=10),
        # a training step of the differentiable projector on a batch of volumes
        _case("autograd3d_128", "step", "joseph", "f32", "both", "128,128,128", "192,192", 180, volumes=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: 2D 64..512, 3D 32..256 (voxel projectors 32..128, FP64 ones
    ..96), axes up to a quarter apart, detectors about as wide as the rotating volume."""
    kind = rng.choice(["project"] * 7 + ["cgls", "batch", "step"])  # FP32 CGLS stays comparable for few iterations
    if kind == "batch":
        lo = _log_int(rng, 64, 160)
        return _case("", kind, "joseph", "f32", "both", "%d,%d" % (lo, _log_int(rng, lo + 32, 400)), "0",
                     rng.randrange(90, 361), problems=rng.randrange(4, 65), iterations=rng.randrange(5, 21))
    method = rng.choice(["joseph"] * 4 + ["siddon"] * 2 + ["blob", "bspline", "pcblob", "pcbspline"])
    if kind in ("step", "cgls"):
        method = "joseph" if kind == "step" else rng.choice(["joseph", "joseph", "siddon"])
    dim = rng.choice([2, 3, 3]) if kind != "step" else 3
    dtype = rng.choice(["f32"] * 3 + ["f64"] + ([] if method == "siddon" else ["bf16"]))
    if kind != "project":
        dtype = "f32"
    top = 512 if dim == 2 else 256
    if dim == 3 and (method not in ("joseph", "siddon") or kind != "project"):
        top = 96 if dtype == "f64" else 128
    n = _log_int(rng, 64 if dim == 2 else 32, top)
    vol = [max(16, min(top, int(n * rng.uniform(0.75, 1.25)))) for _ in range(dim)]
    wide = math.hypot(vol[0], vol[-1]) * MAGNIFICATION  # the turning axes: x and the last
    det = [int(wide * rng.uniform(0.95, 1.1)) + 1]
    if dim == 3:
        det.append(int(vol[1] * MAGNIFICATION * rng.uniform(0.95, 1.3)) + 1)
    poses = max(24, int(max(vol) * rng.uniform(0.6, 1.4)))
    curved = method in ("joseph", "siddon") and kind == "project" and rng.random() < 0.15
    way = rng.choice(["forward", "adjoint", "both"]) if kind == "project" else "both"
    return _case("", kind, method, dtype, way, ",".join(map(str, vol)), ",".join(map(str, det)), poses,
                 arc=0.02 if curved else 0.0, iterations=rng.randrange(2, 4) if kind == "cgls" else 0,
                 volumes=rng.randrange(2, 5) if kind == "step" else 0)


# ---- inputs ------------------------------------------------------------------------------------


def _ints(text):
    return [int(v) for v in text.split(",")]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _volume(shape, seed, dtype):
    """An iterate of a reconstruction: 12 random ellipsoids, and noise of 1 % everywhere."""
    g = np.random.default_rng(seed)
    x = 0.01 * torch.randn(shape, device="cuda", generator=_generator(seed))
    axes = [((torch.arange(n, device="cuda", dtype=torch.float32) + 0.5) / n * 2 - 1).reshape(
        [-1 if i == k else 1 for k in range(len(shape))]) for i, n in enumerate(shape)]
    for _ in range(12):
        amp, q = float(g.uniform(0.1, 1.0)), 0.0
        for a in axes:
            q = q + ((a - float(g.uniform(-0.5, 0.5))) / float(g.uniform(0.1, 0.45))) ** 2
        x += amp * (q <= 1.0)
    return x.to(TORCH[dtype])


def _sinogram(shape, seed, dtype):
    """Line integrals of a centred object with its detail, and noise of 1 %."""
    r = 0.0
    for n in shape[1:]:
        a = (torch.arange(n, device="cuda", dtype=torch.float32) + 0.5) / n * 2 - 1
        r = r * 1.0 + a * a if isinstance(r, float) else r[:, None] + a * a
    body = torch.sqrt(torch.clamp(1.0 - r, min=0.0))
    scale = max(shape[1:]) / 2.0
    g = _generator(seed)
    y = body * (1.0 + 0.2 * torch.rand(shape, device="cuda", generator=g))
    y += 0.01 * torch.randn(shape, device="cuda", generator=g)
    return (scale * y).to(TORCH[dtype])


def _descriptors(case):
    vol, det = _ints(case["vol"]), _ints(case["det"])
    vd = E.VolumeDescriptor(vol)
    n = float(max(vol))
    if case["arc"]:
        dd = E.CurvedCircleTrajectoryGenerator.createTrajectory(case["poses"], vd, 360, 100 * n, 5 * n, case["arc"],
                                                                detectorSize=det)
    else:
        dd = E.CircleTrajectoryGenerator.createTrajectory(case["poses"], vd, 360, 100 * n, 5 * n, detectorSize=det)
    return vd, dd


def _problem_descriptors(case):
    """The uneven 2D problems of a batch: sizes, numbers of poses and start angles. They are the
    case's own (not the seed's), so that every seed has the same amount of work."""
    lo, hi = _ints(case["vol"])
    g = np.random.default_rng(case["problems"] * 1000 + case["iterations"])
    out = []
    for _ in range(case["problems"]):
        n = int(round(math.exp(g.uniform(math.log(lo), math.log(hi)))))
        poses = int(g.integers(case["poses"] // 4, case["poses"] + 1))
        start = float(g.uniform(0, 360))
        vd = E.VolumeDescriptor([n, n])
        det = int(n * math.sqrt(2.0))
        angles = np.deg2rad(start + np.linspace(0, 360, poses)).astype(np.float32)
        geoms = [E.Geometry(100.0 * n, 5.0 * n, vd, [det], float(a)) for a in angles]
        out.append((vd, E.PlanarDetectorDescriptor([det, poses], geoms)))
    return out


def _inputs(case, seed, vd, dd):
    x = _volume(vd.shape, seed, case["dtype"]) if case["way"] != "adjoint" else None
    y = _sinogram(dd.shape, seed, case["dtype"]) if case["way"] != "forward" else None
    return x, y


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        dds = _problem_descriptors(case)
        batch = E.ProjectorBatch([E.JosephsMethodCUDA(vd, dd) for vd, dd in dds])
        b = batch.pack([_sinogram(dd.shape, seed + 7 * j, "f32") for j, (_, dd) in enumerate(dds)],
                       adjoint_space=True)
        return {"case": case, "op": batch, "y": b}
    vd, dd = _descriptors(case)
    op = CLASSES[case["method"]](vd, dd, dtype=DTYPES[case["dtype"]])
    if kind == "step":
        x = torch.stack([_volume(vd.shape, seed + i, "f32") for i in range(case["volumes"])])
        y = torch.stack([_sinogram(dd.shape, seed + i, "f32") for i in range(case["volumes"])])
        project(op, x)  # a training loop keeps the operator's batch from its first step on
        return {"case": case, "op": op, "x": x, "y": y}
    x, y = _inputs(case, seed, vd, dd)
    return {"case": case, "op": op, "x": x, "y": y}


def _total_variation(v):
    dz = v[:, 1:, :-1, :-1] - v[:, :-1, :-1, :-1]
    dy = v[:, :-1, 1:, :-1] - v[:, :-1, :-1, :-1]
    dx = v[:, :-1, :-1, 1:] - v[:, :-1, :-1, :-1]
    return torch.sqrt(dx * dx + dy * dy + dz * dz + 1e-8).sum()


def run(state):
    case, op = state["case"], state["op"]
    if case["kind"] == "project":
        out = {}
        if case["way"] != "adjoint":
            out["sinogram"] = op.apply(state["x"])
        if case["way"] != "forward":
            out["volume"] = op.applyAdjoint(state["y"])
        return out
    if case["kind"] == "step":
        x = state["x"].detach().requires_grad_(True)
        r = project(op, x) - state["y"]
        loss = 0.5 * (r * r).sum() + LAMBDA_TV * _total_variation(x)
        loss.backward()
        return {"gradient": x.grad, "volume": torch.sub(x.detach(), x.grad, alpha=STEP)}
    if case["kind"] == "batch":
        solver = E.APGD(op, state["y"], prox=E.ProximalL1(LAMBDA_L1), graph=True)
    else:
        solver = E.CGLS(op, state["y"], tol=0.0)
    return {"volume": solver.solve(case["iterations"])}


# ---- what a pass cannot do without -------------------------------------------------------------


def _pass_work(method, vol, det, poses, size):
    """(bytes, operations) of one projection: volume and sinogram once, and per ray sample (voxel
    crossing, footprint tap) the operations of its interpolation and sum. The rays of a pose meet
    a plane of voxels with MAGNIFICATION^(dim - 1) rays a voxel, and the planes of their driving
    axis at 0.9 of that on average."""
    dim, nvox = len(vol), float(np.prod(vol))
    samples = 0.9 * poses * nvox * MAGNIFICATION ** (dim - 1)
    if method in SUPPORT:
        taps = poses * nvox * (2 * SUPPORT[method] * MAGNIFICATION) ** (dim - 1)
        flops = 10 * taps
    elif method == "siddon":
        flops = 3 * (1.4 if dim == 3 else 1.3) * samples
    else:
        flops = (15 if dim == 3 else 6) * samples
    return size * (nvox + float(np.prod(det)) * poses), flops


def work(case):
    size = {"f32": 4, "f64": 8, "bf16": 2}[case["dtype"]]
    if case["kind"] == "batch":
        lo, hi = _ints(case["vol"])
        g = np.random.default_rng(case["problems"] * 1000 + case["iterations"])
        total = [0.0, 0.0]
        for _ in range(case["problems"]):
            n = int(round(math.exp(g.uniform(math.log(lo), math.log(hi)))))
            poses = int(g.integers(case["poses"] // 4, case["poses"] + 1))
            g.uniform(0, 360)
            b, f = _pass_work("joseph", [n, n], [int(n * math.sqrt(2.0))], poses, size)
            total = [total[0] + b, total[1] + f]
        passes = 2 * case["iterations"] + 13  # with A^T b and the six of the step length
        return {"bytes": passes * total[0], "flops": passes * total[1]}
    b, f = _pass_work(case["method"], _ints(case["vol"]), _ints(case["det"]), case["poses"], size)
    passes = {"project": 2 if case["way"] == "both" else 1, "cgls": 2 * case["iterations"] + 1,
              "step": 2 * max(1, case["volumes"])}[case["kind"]]
    return {"bytes": passes * b, "flops": passes * f}


# ---- the same in 64 bits -----------------------------------------------------------------------
# elsa's geometry is single precision for every data type: the pose matrices (read from the
# descriptors) and the ray, crossing or footprint set-up below are FP32 by definition and are
# formed in FP32 here too; everything from the sample points on is 64-bit.

CHUNK = 24_000_000  # samples held at once


def _poses(dd, dim):
    """Per pose, as the matrices' columns: Pinv (dim+1 x dim), C, P, ext (dim x dim+1), sdd."""
    f = lambda a: torch.tensor(np.stack(a), dtype=torch.float32, device="cuda")  # noqa: E731
    g = dd.getGeometry()
    return (f([p.getInverseProjectionMatrix() for p in g]), f([p.getCameraCenter() for p in g]),
            f([p.getProjectionMatrix() for p in g]), f([p.getExtrinsicMatrix() for p in g]),
            f([np.float32(p.getSourceDetectorDistance()) for p in g]))


def _rays(dd, poses, k0, k1, dim):
    """Origins and directions (FP32) of the rays of poses k0 <= k < k1, u fastest."""
    pinv, c = poses[0][k0:k1], poses[1][k0:k1]
    n = [int(v) for v in dd.getNumberOfCoefficientsPerDimension()]
    if isinstance(dd, E.CurvedDetectorDescriptor):
        h = torch.tensor(dd.getPlanarCoords(), device="cuda").reshape(-1, dim - 1)
        cols = [h[:, i] for i in range(dim - 1)]
    else:
        u = torch.arange(n[0], device="cuda", dtype=torch.float32) + 0.5
        cols = [u]
        if dim == 3:
            v = torch.arange(n[1], device="cuda", dtype=torch.float32) + 0.5
            cols = [u.repeat(n[1]), v.repeat_interleave(n[0])]
    d, n2 = [], None
    for i in range(dim):
        acc = pinv[:, i, 0, None] * cols[0]
        for j in range(1, dim - 1):
            acc = acc + pinv[:, i, j, None] * cols[j]
        acc = acc + pinv[:, i, dim - 1, None]
        d.append(acc.reshape(-1))
        n2 = d[i] * d[i] if n2 is None else n2 + d[i] * d[i]
    norm = torch.sqrt(n2)
    pixels = d[0].numel() // (k1 - k0)
    return [c[:, i].repeat_interleave(pixels) for i in range(dim)], [v / norm for v in d]


def _box(o, d, vol):
    """Entry and exit parameters of [0, vol) and whether the ray meets it."""
    tmin = tmax = None
    for i in range(len(vol)):
        inv = 1.0 / d[i]
        t1, t2 = (0.0 - o[i]) * inv, (float(vol[i]) - o[i]) * inv
        near, far = torch.where(inv >= 0, t1, t2), torch.where(inv >= 0, t2, t1)
        tmin = near if i == 0 else torch.where(near.isnan() | (near < tmin), tmin, near)
        tmax = far if i == 0 else torch.where(far.isnan() | (far > tmax), tmax, far)
    return tmin, tmax, (tmax >= torch.clamp(tmin, min=0.0)) & ~((tmin == 0) & (tmax == 0))


def _clip(v, hi):
    return torch.clamp(v, min=0.0, max=float(hi))


def _pick(v, axis):
    return torch.stack(v).gather(0, axis[None])[0]


def _joseph_rays(o, d, vol):
    """Sample 0, step, number of samples and step length of every ray (elsa's driving-direction
    traversal, in FP32), and its driving axis."""
    dim = len(vol)
    size = [v.abs() for v in d]
    axis = torch.where(size[1] > size[0], 1, 0)
    big = torch.maximum(size[0], size[1])
    if dim == 3:
        axis = torch.where(size[2] > big, 2, axis)
        big = torch.maximum(big, size[2])
    tmin, tmax, hit = _box(o, d, vol)
    cur = [_clip(o[i] + tmin * d[i], vol[i]) for i in range(dim)]
    end = [_clip(o[i] + tmax * d[i], vol[i]) for i in range(dim)]
    step = [v / big for v in d]
    ca = _pick(cur, axis)
    ahead = 0.5 - (ca - torch.floor(ca))
    s = torch.sign(_pick(step, axis))
    cur = [cur[i] + step[i] * ahead * s for i in range(dim)]
    snapped = torch.floor(_pick(cur, axis)) + 0.5
    n = torch.ceil((_pick(end, axis) - snapped).abs())
    n = torch.where(hit, n, torch.zeros_like(n)).long()
    n2 = step[0] * step[0] + (step[1] * step[1] + step[2] * step[2]) if dim == 3 else \
        step[0] * step[0] + step[1] * step[1]
    first = (snapped - 0.5).long()
    return axis, cur, step, first, torch.where(s < 0, -1, 1), n, torch.sqrt(n2).double()


def _groups(rays, per_ray):
    per = max(1, CHUNK // max(1, per_ray))
    for i in range(0, rays.numel(), per):
        yield rays[i:i + per]


def _strides(vol, pad):
    s, out = 1, []
    for n in vol:
        out.append(s)
        s *= n + 2 * pad
    return out, s


def _joseph(vd, dd, data, adjoint, poses=None):
    """Joseph's method in 64 bits: linear interpolation at the FP32 sample points."""
    vol = [int(v) for v in vd.getNumberOfCoefficientsPerDimension()]
    dim = len(vol)
    poses = poses or _poses(dd, dim)
    stride, total = _strides(vol, 1)
    padded = torch.zeros(tuple(n + 2 for n in vd.shape), dtype=torch.float64, device="cuda")
    inner = padded[tuple(slice(1, -1) for _ in vol)]
    if not adjoint:
        inner.copy_(data)
    flat = padded.reshape(-1)
    nposes, pixels = dd.shape[0], int(np.prod(dd.shape[1:]))
    sino = data.reshape(-1).double() if adjoint else torch.zeros(nposes * pixels, dtype=torch.float64, device="cuda")
    group = max(1, 2_000_000 // pixels)
    for k0 in range(0, nposes, group):
        k1 = min(nposes, k0 + group)
        o, d = _rays(dd, poses, k0, k1, dim)
        axis, cur, step, first, sign, n, length = _joseph_rays(o, d, vol)
        for a in range(dim):
            rays = torch.nonzero((axis == a) & (n > 0)).reshape(-1)
            for r in _groups(rays, vol[a]):
                s = torch.arange(int(n[r].max()), device="cuda")[None]
                plane = first[r][:, None] + s * sign[r][:, None]
                ok = (s < n[r][:, None]) & (plane >= 0) & (plane < vol[a])
                at = (torch.clamp(plane, 0, vol[a] - 1) + 1) * stride[a]
                w, lows = [], []
                for i in [i for i in range(dim) if i != a]:
                    q = (cur[i][r].double()[:, None] + s * step[i][r].double()[:, None]).float().double() - 0.5
                    low = torch.floor(q)
                    w.append(q - low)
                    lows.append(i)
                    at = at + (torch.clamp(low, -1, vol[i] - 1).long() + 1) * stride[i]
                if adjoint:
                    base = torch.where(ok, (sino[k0 * pixels + r] * length[r])[:, None], 0.0)
                else:
                    acc = 0.0
                for corner in range(1 << (dim - 1)):
                    wt, idx = 1.0, at
                    for j, i in enumerate(lows):
                        up = (corner >> j) & 1
                        wt = wt * (w[j] if up else 1.0 - w[j])
                        idx = idx + up * stride[i]
                    if adjoint:
                        flat.index_add_(0, idx.reshape(-1), (wt * base).reshape(-1))
                    else:
                        acc = acc + wt * flat[idx]
                if not adjoint:
                    sino[k0 * pixels + r] = (acc * ok).sum(1) * length[r]
    return inner.clone() if adjoint else sino.reshape(dd.shape)


def _siddon(vd, dd, data, adjoint, poses=None):
    """Siddon's method in 64 bits from the FP32 entry voxel and crossing parameters T0 + k dt: per
    plane of the driving axis at most one crossing of each other axis."""
    vol = [int(v) for v in vd.getNumberOfCoefficientsPerDimension()]
    dim = len(vol)
    poses = poses or _poses(dd, dim)
    stride, total = _strides(vol, 0)
    flat = torch.zeros(total, dtype=torch.float64, device="cuda") if adjoint else data.reshape(-1).double()
    nposes, pixels = dd.shape[0], int(np.prod(dd.shape[1:]))
    sino = data.reshape(-1).double() if adjoint else torch.zeros(nposes * pixels, dtype=torch.float64, device="cuda")
    group = max(1, 2_000_000 // pixels)
    for k0 in range(0, nposes, group):
        k1 = min(nposes, k0 + group)
        o, d = _rays(dd, poses, k0, k1, dim)
        tmin, _, hit = _box(o, d, vol)
        cur, t0, dt, st = [], [], [], []
        for i in range(dim):
            e = _clip(o[i] + tmin * d[i], vol[i])
            sgn = torch.sign(d[i])
            c = torch.floor(e)
            c = torch.where((c == e) & (sgn < 0), c - 1, c)
            hit = hit & (c >= 0) & (c < vol[i])
            moves = d[i].abs() > 1.1920928955078125e-07
            far = torch.full_like(e, math.inf)
            dt.append(torch.where(moves, sgn / d[i], far).double())
            t0.append(torch.where(moves, (torch.where(d[i] > 0, c + 1, c) - e) / d[i], far).double())
            st.append(torch.where(moves, sgn, torch.zeros_like(sgn)).long())
            cur.append(c.long())
        size = [v.abs() for v in d]
        axis = torch.where(size[1] > size[0], 1, 0)
        if dim == 3:
            axis = torch.where(size[2] > torch.maximum(size[0], size[1]), 2, axis)
        for a in range(dim):
            rays = torch.nonzero((axis == a) & hit).reshape(-1)
            for r in _groups(rays, 2 * vol[a]):
                k = torch.arange(vol[a], device="cuda")[None]
                t_out = t0[a][r][:, None] + k * dt[a][r][:, None]
                t_in = torch.where(k == 0, 0.0, t_out - dt[a][r][:, None])
                plane = cur[a][r][:, None] + k * st[a][r][:, None]
                ok = (plane >= 0) & (plane < vol[a])
                cross, counts, others = [], [], [i for i in range(dim) if i != a]
                for i in others:
                    m = torch.floor((t_in - t0[i][r][:, None]) / dt[i][r][:, None]) + 1
                    m = torch.where(torch.isfinite(dt[i][r])[:, None], torch.clamp(m, min=0.0), 0.0)
                    cross.append(torch.where(torch.isfinite(dt[i][r])[:, None],
                                             t0[i][r][:, None] + m * torch.nan_to_num(dt[i][r], posinf=0.0)[:, None],
                                             math.inf))
                    counts.append(m.long())
                edges = torch.sort(torch.stack([torch.minimum(torch.maximum(c, t_in), t_out) for c in cross]), 0)[0]
                edges = [t_in] + list(edges) + [t_out]
                acc = 0.0
                for lo, hi in zip(edges[:-1], edges[1:]):
                    mid, inside, idx = 0.5 * (lo + hi), ok, torch.clamp(plane, 0, vol[a] - 1) * stride[a]
                    for i, c, m in zip(others, cross, counts):
                        x = cur[i][r][:, None] + (m + (mid > c)) * st[i][r][:, None]
                        inside = inside & (x >= 0) & (x < vol[i])
                        idx = idx + torch.clamp(x, 0, vol[i] - 1) * stride[i]
                    w = torch.where(inside, hi - lo, 0.0)
                    if adjoint:
                        flat.index_add_(0, idx.reshape(-1), (w * sino[k0 * pixels + r][:, None]).reshape(-1))
                    else:
                        acc = acc + w * flat[idx]
                if not adjoint:
                    sino[k0 * pixels + r] = acc.sum(1)
    return flat.reshape(vd.shape) if adjoint else sino.reshape(dd.shape)


def _table(case, dim):
    """The projected basis function's table and its support, as the projector holds it."""
    kind, dtype = case["method"], np.float64 if case["dtype"] == "f64" else np.float32
    if kind == "blob":
        t, s = E.projectors.blob_lut(dtype=dtype)
    elif kind == "bspline":
        t, s = E.projectors.bspline_lut(dim, dtype=dtype)
    elif kind == "pcblob":
        t, s = E.projectors.blob_derivative_lut(dtype=dtype, normalized=dim == 3)
    else:
        t, s = E.projectors.bspline_derivative_lut(dim, dtype=dtype, normalized=dim == 3)
    return torch.tensor(t, device="cuda").double(), float(np.float32(s))


def _voxel(case, vd, dd, data, adjoint):
    """The voxel-driven projectors in 64 bits from the FP32 footprint centres and scalings."""
    vol = [int(v) for v in vd.getNumberOfCoefficientsPerDimension()]
    det = [int(v) for v in dd.getNumberOfCoefficientsPerDimension()][:-1]
    dim = len(vol)
    table, support = _table(case, dim)
    table = torch.cat([table, torch.zeros(1, dtype=torch.float64, device="cuda")])
    last = table.numel() - 2
    _, _, P, ext, sdd = _poses(dd, dim)
    ax = [torch.arange(n, device="cuda", dtype=torch.float32) + 0.5 for n in vol]
    grid = [g.reshape(-1) for g in torch.meshgrid(*ax[::-1], indexing="ij")][::-1]
    nposes, pixels = dd.shape[0], int(np.prod(dd.shape[1:]))
    sino = torch.zeros(nposes, pixels, dtype=torch.float64, device="cuda") if not adjoint else \
        data.reshape(nposes, pixels).double()
    out = torch.zeros(grid[0].numel(), dtype=torch.float64, device="cuda") if adjoint else data.reshape(-1).double()
    for k in range(nposes):
        def apply(M, i):
            acc = M[k, i, 0] * grid[0]
            for j in range(1, dim):
                acc = acc + M[k, i, j] * grid[j]
            return acc + M[k, i, dim]

        pc, ce = [apply(P, i) for i in range(dim)], [apply(ext, i) for i in range(dim)]
        n2 = ce[0] * ce[0]
        for i in range(1, dim):
            n2 = n2 + ce[i] * ce[i]
        scaling = sdd[k] / torch.sqrt(n2)
        reach = scaling * np.float32(support)
        centre = [pc[i] / pc[dim - 1] - 0.5 for i in range(dim - 1)]
        low = [torch.ceil(c - reach) for c in centre]
        high = [torch.floor(c + reach) for c in centre]
        wide = [int((h - l).max()) + 1 for l, h in zip(low, high)] + ([1] if dim == 2 else [])
        s64, c64 = scaling.double(), [c.double() for c in centre]
        for b in range(wide[1]):
            j = low[1] + b if dim == 3 else None
            for a in range(wide[0]):
                i = low[0] + a
                ok = (i <= high[0]) & (i >= 0) & (i < det[0])
                d0 = (c64[0] - i.double()) / s64
                dist = d0.abs()
                pix = torch.clamp(i, 0, det[0] - 1).long()
                if dim == 3:
                    ok = ok & (j <= high[1]) & (j >= 0) & (j < det[1])
                    d1 = (c64[1] - j.double()) / s64
                    dist = torch.sqrt(d0 * d0 + d1 * d1)
                    pix = pix + torch.clamp(j, 0, det[1] - 1).long() * det[0]
                index = dist / support * last
                ok = ok & (index <= last)
                at = torch.clamp(torch.floor(index), max=float(last)).long()
                t = index - at
                w = table[at] * (1 - t) + table[torch.clamp(at + 1, max=last)] * t
                if case["method"].startswith("pc"):
                    w = w * (torch.sign(d0) if dim == 2 else d0)
                w = torch.where(ok, w, 0.0)
                if adjoint:
                    out += w * sino[k][pix]
                else:
                    sino[k].index_add_(0, pix, w * out)
    return out.reshape(vd.shape) if adjoint else sino.reshape(dd.shape)


def _solve(method, vd, dd, b, iterations):
    A = _joseph if method == "joseph" else _siddon
    poses = _poses(dd, vd.getNumberOfDimensions())
    x, s = torch.zeros(vd.shape, dtype=torch.float64, device="cuda"), b.double().reshape(dd.shape)
    r = A(vd, dd, s, True, poses)
    c, kold = r.clone(), (r * r).sum()
    for _ in range(iterations):
        q = A(vd, dd, c, False, poses)
        alpha = kold / (q * q).sum()
        x, s = x + alpha * c, s - alpha * q
        r = A(vd, dd, s, True, poses)
        k = (r * r).sum()
        c, kold = r + k / kold * c, k
    return x


def _fista(vd, dd, b, iterations):
    poses = _poses(dd, vd.getNumberOfDimensions())
    normal = lambda v: _joseph(vd, dd, _joseph(vd, dd, v, False, poses), True, poses)  # noqa: E731
    u = torch.ones(vd.shape, dtype=torch.float64, device="cuda")
    for _ in range(5):
        u = normal(u)
        u = u / torch.linalg.norm(u)
    mu = 0.45 / ((u * normal(u)).sum() / torch.linalg.norm(u))
    atb = _joseph(vd, dd, b.double().reshape(dd.shape), True, poses)
    x = y = torch.zeros(vd.shape, dtype=torch.float64, device="cuda")
    t = 1.0
    for _ in range(iterations):
        z = y - mu * (normal(y) - atb)
        new = torch.sign(z) * torch.clamp(z.abs() - mu * LAMBDA_L1, min=0.0)
        t_new = (1.0 + math.sqrt(1.0 + 4.0 * t * t)) / 2.0
        y = new + (t - 1.0) / t_new * (new - x)
        x, t = new, t_new
    return x


def exact(case, seed):
    w = work(case)
    if w["flops"] > 5.0e11:  # about 20 seconds
        return None
    kind = case["kind"]
    if kind == "batch":
        return {"volume": torch.cat([_fista(vd, dd, _sinogram(dd.shape, seed + 7 * j, "f32"),
                                            case["iterations"]).reshape(-1)
                                     for j, (vd, dd) in enumerate(_problem_descriptors(case))])}
    vd, dd = _descriptors(case)
    if kind == "cgls":
        return {"volume": _solve(case["method"], vd, dd, _inputs(case, seed, vd, dd)[1], case["iterations"])}
    if kind == "step":
        poses = _poses(dd, 3)
        xs = [_volume(vd.shape, seed + i, "f32").double() for i in range(case["volumes"])]
        grads = []
        for i, x in enumerate(xs):
            r = _joseph(vd, dd, x, False, poses) - _sinogram(dd.shape, seed + i, "f32").double()
            v = x[None].clone().requires_grad_(True)
            tv, = torch.autograd.grad(LAMBDA_TV * _total_variation(v), v)
            grads.append(_joseph(vd, dd, r, True, poses) + tv[0])
        g, x = torch.stack(grads), torch.stack(xs)
        return {"gradient": g, "volume": x - STEP * g}
    x, y = _inputs(case, seed, vd, dd)
    A = {"joseph": _joseph, "siddon": _siddon}.get(case["method"], lambda *a: _voxel(case, *a))
    out = {}
    if case["way"] != "adjoint":
        out["sinogram"] = A(vd, dd, x.double(), False)
    if case["way"] != "forward":
        out["volume"] = A(vd, dd, y.double(), True)
    return out
