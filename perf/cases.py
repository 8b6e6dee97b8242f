"""The work a user has this engine do, as cases that can be timed and compared.

Inputs are seeded phantoms (ellipsoids of three tissue classes, smoothed, with noise; the moving
image seen through a random affine and a smooth displacement), made on the GPU with operations that
give the same bits every time, and rounded to f32 as scanner volumes are. The kinds:

mi_value     one Mattes value of a linear-stage level (the line search's plain probe)
mi_values    four values in one call (the line search's speculative probes)
mi_gradient  one value with its parameter derivative (a conjugate-gradient step)
cc           the neighbourhood cross-correlation pair of a SyN iteration on the caller's device buffers
syn          SyN iterations on images in HBM from a known affine, fields brought to the host
register     a full normalisation, host volumes in, affine and fields out
resident     the same from volumes already in HBM
batch        several subjects against one template, all channels in HBM
linear       many rigid and affine fits side by side
"""
from __future__ import annotations

import ctypes as C
import functools
import math

import numpy as np
import torch

from fastwarp_amd import register as reg
from fastwarp_amd._abi import Affine, Grid, LinearTransform, MiBinning
from fastwarp_amd.backend import FW_OK, HipBackend, MiLevel, RegError, lib

T1 = (0.0, 0.3, 0.6, 1.0)
T2 = (1.0, 0.7, 0.4, 0.1)
EPS = 2.220446049250313e-16


# ------------------------------------------------------------------------------------- the cases

def listed():
    return [
        # a coarse level of a 1 mm linear stage (shrink 8 of 182 x 218 x 182, 25 % of the level's
        # voxels sampled): about 800 such calls a registration, each waiting for the one before
        dict(name="mi_value_coarse", kind="mi_value", nx=182, ny=218, nz=182, spacing=1.0, shrink=8, bins=32, affine=False),
        # the line search's probes on a middle level (shrink 2): two golden-section steps in a call
        dict(name="mi_probes_middle", kind="mi_values", nx=182, ny=218, nz=182, spacing=1.0, shrink=2, bins=32, affine=False),
        # a gradient of the affine stage at full resolution, 1.8 million samples
        dict(name="mi_gradient_fine", kind="mi_gradient", nx=182, ny=218, nz=182, spacing=1.0, shrink=1, bins=32, affine=True),
        # the CC pair on a middle level of the pyramid (shrink 4 of 1 mm), odd sizes
        dict(name="cc_middle", kind="cc", nx=45, ny=54, nz=45, spacing=4.0, radius=4, oblique=False),
        # the CC pair at full 1 mm resolution
        dict(name="cc_fine", kind="cc", nx=182, ny=218, nz=182, spacing=1.0, radius=4, oblique=False),
        # a whole SyN stage at 2 mm, three levels, after a linear stage run elsewhere
        dict(name="syn_2mm", kind="syn", nx=96, ny=112, nz=96, spacing=2.0, levels="40x20x10", channels=1, mixed=False, masks=False),
        # two channels, CC and Mattes, inside brain masks: the multi-modal stage
        dict(name="syn_masked_mixed", kind="syn", nx=80, ny=95, nz=79, spacing=2.0, levels="10x5", channels=2, mixed=True, masks=True),
        # the finest level of the 1 mm cohort plan: 20 iterations at full resolution
        dict(name="syn_1mm_finest", kind="syn", nx=182, ny=218, nz=182, spacing=1.0, levels="20", channels=1, mixed=False, masks=False),
        # a 2 mm normalisation from host volumes, the subject on its own anisotropic grid
        dict(name="register_2mm", kind="register", nx=96, ny=112, nz=96, spacing=2.0, mx=90, my=101, mz=71, channels=1, plan="2mm"),
        # the headline: a 1 mm normalisation with the cohort plan, volumes in HBM
        dict(name="register_1mm", kind="resident", nx=182, ny=218, nz=182, spacing=1.0, channels=1, plan="cohort"),
        # a small two-channel cohort against one 2 mm template
        dict(name="batch_2mm", kind="batch", nx=91, ny=109, nz=91, spacing=2.0, subjects=4, channels=2, plan="2mm"),
        # linear fits of uneven sizes and spacings side by side, as a motion or intake queue has them
        dict(name="linear_fits", kind="linear", fits=8, least=64, most=144),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mi_value", "mi_values", "mi_gradient", "cc", "cc", "syn", "syn", "register", "resident", "batch", "linear"])
    if kind.startswith("mi_"):
        shrink = rng.choice([8, 4, 2, 1])
        return dict(kind=kind, nx=rng.randint(80, 190), ny=rng.randint(80, 220), nz=rng.randint(60, 190), shrink=shrink,
                    spacing=rng.choice([1.0, 1.5, 2.0]), bins=rng.choice([32, 32, 32, 24, 48]), affine=rng.random() < 0.5)
    if kind == "cc":
        return dict(kind=kind, nx=_log(rng, 18, 200), ny=_log(rng, 18, 220), nz=_log(rng, 9, 190), spacing=rng.choice([1.0, 2.0, 4.0]),
                    radius=rng.choice([4, 4, 4, 3, 2]), oblique=rng.random() < 0.25)
    if kind == "syn":
        channels = rng.choice([1, 1, 2])
        return dict(kind=kind, nx=rng.randint(40, 130), ny=rng.randint(40, 130), nz=rng.randint(40, 130), spacing=rng.choice([1.0, 1.5, 2.0]),
                    levels=rng.choice(["40x20x10", "20x10", "12", "10x5"]), channels=channels, mixed=channels == 2 and rng.random() < 0.5,
                    masks=rng.random() < 0.3)
    if kind == "register":
        return dict(kind=kind, nx=rng.randint(64, 120), ny=rng.randint(64, 120), nz=rng.randint(64, 110), spacing=2.0, mx=rng.randint(64, 120),
                    my=rng.randint(64, 120), mz=rng.randint(48, 100), channels=rng.choice([1, 1, 2]), plan="2mm")
    if kind == "resident":
        return dict(kind=kind, nx=rng.randint(64, 150), ny=rng.randint(64, 150), nz=rng.randint(64, 150), spacing=rng.choice([1.0, 1.5, 2.0]),
                    channels=rng.choice([1, 1, 2]), plan=rng.choice(["2mm", "cohort"]))
    if kind == "batch":
        return dict(kind=kind, nx=rng.randint(56, 96), ny=rng.randint(56, 112), nz=rng.randint(56, 96), spacing=2.0, subjects=rng.randint(2, 4),
                    channels=rng.choice([1, 2]), plan="2mm")
    least = rng.randint(48, 80)
    return dict(kind="linear", fits=rng.randint(2, 8), least=least, most=least + rng.randint(10, 60))


# ------------------------------------------------------------------------------------- phantoms

def _gauss(v, sigma):
    """Separable Gaussian along the last three axes, edges repeated: shifted sums in a fixed order."""
    r = max(1, int(3.0 * sigma + 0.5))
    w = [math.exp(-0.5 * (t / sigma) ** 2) for t in range(-r, r + 1)]
    s = sum(w)
    for ax in (-1, -2, -3):
        n = v.shape[ax]
        idx = torch.arange(n, device=v.device)
        out = torch.zeros_like(v)
        for t in range(-r, r + 1):
            out += (w[t + r] / s) * v.index_select(v.dim() + ax, (idx + t).clamp(0, n - 1))
        v = out
    return v


def _axes(g, dtype=torch.float64):
    nx, ny, nz = g.shape_xyz
    z, y, x = (torch.arange(n, device="cuda", dtype=dtype) for n in (nz, ny, nx))
    return x.view(1, 1, -1), y.view(1, -1, 1), z.view(-1, 1, 1)


def _points(g):
    """The physical points of a grid's voxels, (3, nz, ny, nx) f64."""
    x, y, z = _axes(g)
    d = g.dir_matrix() * np.array(list(g.spacing))
    o = list(g.origin)
    return torch.stack([float(d[a, 0]) * x + float(d[a, 1]) * y + float(d[a, 2]) * z + float(o[a]) for a in range(3)])


def _index(g, p):
    """Continuous indices of physical points (3, ...)."""
    m = np.linalg.inv(g.dir_matrix() * np.array(list(g.spacing)))
    q = [p[a] - float(g.origin[a]) for a in range(3)]
    return torch.stack([float(m[a, 0]) * q[0] + float(m[a, 1]) * q[1] + float(m[a, 2]) * q[2] for a in range(3)])


def _inside(v, c):
    n = (v.shape[2], v.shape[1], v.shape[0])
    ok = torch.ones_like(c[0], dtype=torch.bool)
    for a in range(3):
        ok &= (c[a] >= -0.5) & (c[a] < n[a] - 0.5)
    return ok


def _sample(v, c):
    """Trilinear values of v (nz, ny, nx) at continuous indices c (3, ...), indices clamped to the buffer."""
    nz, ny, nx = v.shape
    flat = v.reshape(-1)
    lo, w = [], []
    for a, n in enumerate((nx, ny, nz)):
        q = c[a].clamp(0, n - 1)
        f = q.floor().clamp(max=n - 1)
        lo.append(f.long())
        w.append(q - f)
    out = torch.zeros_like(c[0])
    for corner in range(8):
        wt, idx = None, []
        for a, n in enumerate((nx, ny, nz)):
            up = (corner >> a) & 1
            f = w[a] if up else 1.0 - w[a]
            wt = f if wt is None else wt * f
            idx.append((lo[a] + up).clamp(max=n - 1))
        out += wt * flat[idx[0] + nx * (idx[1] + ny * idx[2])]
    return out


def _grid(shape, spacing, direction=None):
    spacing = (spacing,) * 3 if isinstance(spacing, (int, float)) else spacing
    origin = np.array([-(n - 1) * s / 2.0 for n, s in zip(shape, spacing)])
    if direction is not None:
        origin = direction @ origin
    return Grid.make(shape, spacing, origin, direction)


def _f32(v):
    return v.float().double()


def _rotation(rng):
    q = rng.normal(size=4)
    w, x, y, z = q / np.linalg.norm(q)
    return np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)],
                     [2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)],
                     [2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]])


def _noise(shape, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).double()


def _fixed(grid, rng, channels):
    """The fixed volumes: forty ellipsoids of three classes painted in order, smoothed, with noise."""
    x, y, z = _axes(grid, torch.float32)
    shape = grid.shape_xyz
    label = torch.zeros(shape[::-1], device="cuda", dtype=torch.long)
    small = min(1.0, min(shape) / 90.0)
    for _ in range(40):
        c = rng.uniform(0.1 * np.array(shape), 0.9 * np.array(shape))
        r = _rotation(rng) / (rng.uniform(4.0, 20.0, size=3) * small)
        tissue = int(rng.integers(0, 4))
        q = 0
        for a in range(3):
            q = q + (float(r[0, a]) * (x - float(c[0])) + float(r[1, a]) * (y - float(c[1])) + float(r[2, a]) * (z - float(c[2]))) ** 2
        label = torch.where(q <= 1.0, tissue, label)
    out = []
    for ch in range(channels):
        table = torch.tensor(T1 if ch == 0 else T2, device="cuda", dtype=torch.float64)
        v = _gauss(table[label], 1.0)
        out.append(_f32(v + 0.02 * _noise(v.shape, rng.integers(1 << 31))))
    return out


def _true_affine(rng, degrees, mm):
    ang = np.deg2rad(rng.uniform(-degrees, degrees, size=3))
    (cx, cy, cz), (sx, sy, sz) = np.cos(ang), np.sin(ang)
    rx = np.array([[1, 0, 0], [0, cx, -sx], [0, sx, cx]])
    ry = np.array([[cy, 0, sy], [0, 1, 0], [-sy, 0, cy]])
    rz = np.array([[cz, -sz, 0], [sz, cz, 0], [0, 0, 1]])
    return rz @ rx @ ry @ np.diag(rng.uniform(0.95, 1.05, size=3)), rng.uniform(-mm, mm, size=3)


def _moving(grid, moving_grid, fixed, rng, degrees=10.0, mm=5.0, bend_mm=4.0):
    """The moving volumes, and the affine that takes moving-grid points to fixed-grid points."""
    mat, trans = _true_affine(rng, degrees, mm)
    p = _points(moving_grid)
    if bend_mm > 0:
        u = _gauss(_noise((3,) + p.shape[1:], rng.integers(1 << 31)), 6.0)
        u *= bend_mm / float(u.square().sum(0).max().sqrt())
        p = p + u
    q = torch.stack([float(mat[a, 0]) * p[0] + float(mat[a, 1]) * p[1] + float(mat[a, 2]) * p[2] + float(trans[a]) for a in range(3)])
    c = _index(grid, q)
    out = []
    for v in fixed:
        m = torch.where(_inside(v, c), _sample(v, c), 0.0)
        out.append(_f32(m.clamp(min=0.0) ** 0.8))
    inv = np.linalg.inv(mat)
    return out, Affine.make(inv, -inv @ trans)


def _host(v):
    return v.reshape(-1).cpu().numpy()


@functools.lru_cache(maxsize=1)
def _backend():
    return HipBackend()


def _plan(case):
    return reg.cohort_plan(case["channels"]) if case["plan"] == "cohort" else reg.plan_2mm(case["channels"])


# ------------------------------------------------------------------------------------- prepare

def _level(case, seed):
    """A linear-stage level: the smoothed moving image, the sample points and their fixed bins."""
    rng = np.random.default_rng(seed)
    g = _grid((case["nx"], case["ny"], case["nz"]), case["spacing"])
    fixed = _fixed(g, rng, 1)
    moving, _ = _moving(g, g, fixed, rng)
    sigma = {8: 3.0, 4: 2.0, 2: 1.0, 1: 0.0}[case["shrink"]]
    f, m = (_f32(_gauss(v[0], sigma)) if sigma else v[0] for v in (fixed, moving))
    # every fourth voxel of the level's grid in raster order, jittered by a third of its spacing
    s = case["shrink"]
    nx, ny, nz = (n // s for n in g.shape_xyz)
    flat = torch.arange(0, nx * ny * nz, 4, device="cuda")
    idx = torch.stack([flat % nx, (flat // nx) % ny, flat // (nx * ny)]).double()
    c = (idx + _noise(idx.shape, rng.integers(1 << 31)) / 3.0) * s + (s - 1) / 2.0
    c = c[:, _inside(f, c)]
    value = _sample(f, c)
    sp = case["spacing"]
    points = torch.stack([c[a] * sp + float(g.origin[a]) for a in range(3)], dim=1).contiguous()
    binning = MiBinning.from_ranges(case["bins"], (float(f.min()), float(f.max())), (float(m.min()), float(m.max())))
    bins = (value / binning.fixed_bin_size - binning.fixed_normalized_min).long().clamp(2, case["bins"] - 3)
    transforms = []
    for _ in range(4):
        mat, trans = _true_affine(rng, 4.0, 3.0)
        if case["affine"]:
            transforms.append(LinearTransform.make(1, list(mat.reshape(-1)) + list(trans)))
        else:
            transforms.append(LinearTransform.make(0, list(np.deg2rad(rng.uniform(-4, 4, size=3))) + list(trans)))
    return g, m, points, bins, binning, transforms


def _prepare_mi(case, seed):
    g, m, points, bins, binning, transforms = _level(case, seed)
    b = _backend()
    level = MiLevel(b, b.upload_image(g, _host(m)), points.cpu().numpy(), bins.int().cpu().numpy().astype(np.uint32), binning)
    return dict(case=case, level=level, transforms=transforms)


def _cc_images(case, seed):
    rng = np.random.default_rng(seed)
    direction = None
    if case["oblique"]:
        a = 0.3
        direction = np.array([[math.cos(a), -math.sin(a), 0], [math.sin(a), math.cos(a), 0], [0, 0, 1.0]])
    g = _grid((case["nx"], case["ny"], case["nz"]), case["spacing"], direction)
    fixed = _fixed(g, rng, 1)
    # as a SyN iteration sees them: the moving image close to the fixed one already
    moving, _ = _moving(g, g, fixed, rng, degrees=2.0, mm=1.0 * case["spacing"], bend_mm=2.0 * case["spacing"])
    return g, fixed[0], moving[0]


def _prepare_cc(case, seed):
    g, f, m = _cc_images(case, seed)
    # the values beside the fields: device memory the caller owns
    out = [torch.zeros((3,) + f.shape, device="cuda") for _ in range(2)] + [torch.zeros(2, device="cuda", dtype=torch.float64)]
    return dict(case=case, grid=g, fixed=f.float().contiguous(), moving=m.float().contiguous(), out=out)


def _ball(grid, share):
    x, y, z = _axes(grid)
    nx, ny, nz = grid.shape_xyz
    q = ((x - (nx - 1) / 2) / (share * nx / 2)) ** 2 + ((y - (ny - 1) / 2) / (share * ny / 2)) ** 2 + ((z - (nz - 1) / 2) / (share * nz / 2)) ** 2
    return (q <= 1.0).double()


def _prepare_syn(case, seed):
    rng = np.random.default_rng(seed)
    b = _backend()
    g = _grid((case["nx"], case["ny"], case["nz"]), case["spacing"])
    fixed = _fixed(g, rng, case["channels"])
    moving, affine = _moving(g, g, fixed, rng)
    # intensities in [0, 1], as a winsorised volume has them
    up = lambda v: b.upload_image(g, _host(_f32(v.clamp(0.0, 1.0))))  # noqa: E731
    plan = reg.cohort_plan(case["channels"])
    its = [int(t) for t in case["levels"].split("x")]
    shrink = [1 << k for k in range(len(its) - 1, -1, -1)]
    plan.set_syn(its, shrink, [float(k) for k in range(len(its) - 1, -1, -1)])
    # a fixed number of iterations: the convergence window never fills
    plan.syn_convergence_threshold = 0.0
    if case["mixed"]:
        plan.syn_channel_metrics[1] = 1
    masks = [b.upload_image(g, _host(_ball(g, s))) if case["masks"] else None for s in (0.9, 0.95)]
    return dict(case=case, backend=b, plan=plan, fixed=[up(v) for v in fixed], moving=[up(v) for v in moving], affine=affine, masks=masks)


def _prepare_register(case, seed):
    rng = np.random.default_rng(seed)
    g = _grid((case["nx"], case["ny"], case["nz"]), case["spacing"])
    size = (case["mx"], case["my"], case["mz"])
    mg = _grid(size, tuple(n * case["spacing"] / k for n, k in zip(g.shape_xyz, size)))
    fixed = _fixed(g, rng, case["channels"])
    moving, _ = _moving(g, mg, fixed, rng)
    return dict(case=case, backend=_backend(), plan=_plan(case), grids=(g, mg), fixed=[_host(v) for v in fixed], moving=[_host(v) for v in moving])


def _prepare_resident(case, seed):
    rng = np.random.default_rng(seed)
    b = _backend()
    g = _grid((case["nx"], case["ny"], case["nz"]), case["spacing"])
    fixed = _fixed(g, rng, case["channels"])
    moving, _ = _moving(g, g, fixed, rng)
    up = lambda v: b.upload_image(g, _host(v))  # noqa: E731
    return dict(case=case, backend=b, plan=_plan(case), fixed=[up(v) for v in fixed], moving=[up(v) for v in moving])


def _prepare_batch(case, seed):
    rng = np.random.default_rng(seed)
    b = _backend()
    g = _grid((case["nx"], case["ny"], case["nz"]), case["spacing"])
    fixed = _fixed(g, rng, case["channels"])
    up = lambda v: b.upload_image(g, _host(v))  # noqa: E731
    moving = [[up(v) for v in _moving(g, g, fixed, rng)[0]] for _ in range(case["subjects"])]
    return dict(case=case, backend=b, plan=_plan(case), fixed=[up(v) for v in fixed], moving=moving)


def _fit_sizes(case):
    """The fits' grids: uneven sizes from `least` to `most` voxels an axis, three spacings."""
    rng = np.random.default_rng(case["fits"] * 1000 + case["least"])
    return [([int(v) for v in rng.integers(case["least"], case["most"] + 1, size=3)], [1.0, 1.5, 2.0][i % 3]) for i in range(case["fits"])]


def _prepare_linear(case, seed):
    rng = np.random.default_rng(seed)
    b = _backend()
    plan = reg.cohort_plan(1)
    plan.run_syn = 0
    fixed, moving = [], []
    for shape, spacing in _fit_sizes(case):
        g = _grid(shape, spacing)
        f = _fixed(g, rng, 1)
        m, _ = _moving(g, g, f, rng, bend_mm=0.0)
        fixed.append(b.upload_image(g, _host(f[0])))
        moving.append(b.upload_image(g, _host(m[0])))
    return dict(case=case, backend=b, plan=plan, fixed=fixed, moving=moving)


def prepare(case, seed):
    kind = case["kind"]
    if kind.startswith("mi_"):
        return _prepare_mi(case, seed)
    return {"cc": _prepare_cc, "syn": _prepare_syn, "register": _prepare_register, "resident": _prepare_resident,
            "batch": _prepare_batch, "linear": _prepare_linear}[kind](case, seed)


# ------------------------------------------------------------------------------------- run

def _affine_out(a):
    return {"matrix": np.array(list(a.matrix)), "translation": np.array(list(a.translation))}


def _resident_out(backend, r):
    return {**_affine_out(r.affine), "forward": backend.download_field(r.forward), "inverse": backend.download_field(r.inverse)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "mi_value":
        return state["level"].value(state["transforms"][0])
    if kind == "mi_values":
        return state["level"].values(state["transforms"])
    if kind == "mi_gradient":
        v, d = state["level"].value_and_derivative(state["transforms"][0])
        return {"value": v, "derivative": d}
    if kind == "cc":
        o = state["out"]
        rc = lib().fw_cc_pair_noalloc(C.byref(state["grid"]), state["fixed"].data_ptr(), state["moving"].data_ptr(), case["radius"],
                                      o[0].data_ptr(), o[1].data_ptr(), o[2].data_ptr(), None)
        if rc != FW_OK:
            raise RegError(rc, lib().fw_last_error(None).decode())
        return o
    b, plan = state["backend"], state["plan"]
    if kind == "syn":
        r = reg.syn_stage(b, plan, state["fixed"], state["moving"], state["affine"], state["masks"][0], state["masks"][1])
        return {"forward": b.download_field(r.forward), "inverse": b.download_field(r.inverse),
                "energy": np.array(list(r.result.syn_last_energy)[: plan.syn_levels])}
    if kind == "register":
        r = reg.register(b, plan, state["grids"][0], state["fixed"], state["grids"][1], state["moving"])
        return {**_affine_out(r.affine), "forward": r.forward, "inverse": r.inverse}
    if kind == "resident":
        return _resident_out(b, reg.register_resident(b, plan, state["fixed"], state["moving"]))
    if kind == "batch":
        return [_resident_out(b, r) for r in reg.register_batch(b, plan, state["fixed"], state["moving"])]
    return [_affine_out(r.affine) for r in reg.linear_batch(b, plan, state["fixed"], state["moving"])]


# ------------------------------------------------------------------------------------- work

def _samples(case):
    s = case["shrink"]
    return (case["nx"] // s) * (case["ny"] // s) * (case["nz"] // s) / 4


def _syn_work(voxels, plan_levels, channels):
    """A SyN iteration reads the images and the four fields of its state and writes the four fields;
    the metric's window sums, the smoothing and the gathers are about 500 operations a voxel."""
    its = sum(n * voxels / s**3 for n, s in plan_levels)
    return its * (96 + 8 * channels), its * (250 * channels + 400)


def _linear_work(voxels, levels):
    """A linear level of either stage takes about 200 metric evaluations; each reads its samples (16
    bytes), a quarter of the level's voxels, and the eight neighbours of each in the moving image
    (at least one value a sample)."""
    e = sum(2 * 200 * voxels / s**3 / 4 for s in levels)
    return e * 20, e * 150


def work(case):
    kind = case["kind"]
    if kind.startswith("mi_"):
        m, k = _samples(case), 4 if kind == "mi_values" else 1
        # the records, the moving image's values (each once at most) and the histogram's cells
        image = 4.0 * min(8 * m, case["nx"] * case["ny"] * case["nz"])
        return {"bytes": 16 * m + image + 8 * k * case["bins"] ** 2, "flops": m * k * 100 * (2 if kind == "mi_gradient" else 1)}
    if kind == "cc":
        n = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": 32 * n, "flops": 150 * n}
    if kind == "linear":
        b = f = 0.0
        for shape, _ in _fit_sizes(case):
            n = float(np.prod(shape))
            wb, wf = _linear_work(n, (8, 4, 2, 1))
            b, f = b + wb + 8 * n, f + wf
        return {"bytes": b, "flops": f}
    n = float(case["nx"] * case["ny"] * case["nz"])
    if kind == "syn":
        its = [int(t) for t in case["levels"].split("x")]
        wb, wf = _syn_work(n, [(t, 1 << k) for k, t in zip(range(len(its) - 1, -1, -1), its)], case["channels"])
        return {"bytes": wb + 24 * n, "flops": wf}
    levels = [(100, 8), (70, 4), (50, 2), (20, 1)] if case["plan"] == "cohort" else [(40, 4), (20, 2), (10, 1)]
    wb, wf = _syn_work(n, levels, case["channels"])
    lb, lf = _linear_work(n, [s for _, s in levels])
    k = case.get("subjects", 1)
    return {"bytes": k * (wb + lb + (24 + 8 * case["channels"]) * n), "flops": k * (wf + lf)}


# ------------------------------------------------------------------------------------- tolerance

def tolerance(case):
    """About four times the difference of two builds that round the CC derivative and the sampled
    coordinates in another order in f32, over the listed cases and fourteen drawn ones. One
    evaluation differs by 7e-8 (values), 3e-6 (gradients) and 4e-8 (CC; on oblique grids the f32
    gradients are 1.3e-6 from f64). In a SyN stage now and then one inversion takes another number
    of steps (a tie at its 0.1 voxel tolerance): 2.5e-3 of the fields, 0.2 of their root mean square
    at one voxel. A linear fit ends within 3e-3 of the other; a registration carries that into its
    fields, 1e-2 to 8e-2 of them, so its tolerance is as wide as one may be."""
    kind = case["kind"]
    if kind in ("mi_value", "mi_values"):
        return {"rel": 2e-6}
    if kind == "mi_gradient":
        return {"rel": 2e-5, "max": 1e-4}
    if kind == "cc":
        return {"rel": 5e-6, "max": 5e-5} if case["oblique"] else {"rel": 2e-7, "max": 2e-6}
    if kind == "syn":
        return {"rel": 1e-2, "max": 0.8}
    if kind == "linear":
        return {"rel": 1.2e-2, "max": 2e-2}
    return {"rel": 0.03, "max": 0.99}


# ------------------------------------------------------------------------------------- exact

def _bspline(u):
    a = u.abs()
    s = a * a
    return torch.where(a < 1, (4 - 6 * s + 3 * s * a) / 6, torch.where(a < 2, (8 - 12 * a + 6 * s - s * a) / 6, 0.0))


def _bspline_d(u):
    r = torch.zeros_like(u)
    r = torch.where((u >= 0) & (u < 1), -2 * u + 1.5 * u * u, r)
    r = torch.where((u > -1) & (u < 0), -2 * u - 1.5 * u * u, r)
    r = torch.where((u >= 1) & (u < 2), -2 + 2 * u - 0.5 * u * u, r)
    return torch.where((u > -2) & (u <= -1), 2 + 2 * u + 0.5 * u * u, r)


def _matrix(t):
    """The matrix of a transform's own part and its translation (the centre is the origin here)."""
    p = list(t.parameters)
    if t.kind == 1:
        return np.array(p[:9]).reshape(3, 3), np.array(p[9:12])
    (cx, cy, cz), (sx, sy, sz) = np.cos(p[:3]), np.sin(p[:3])
    rx = np.array([[1, 0, 0], [0, cx, -sx], [0, sx, cx]])
    ry = np.array([[cy, 0, sy], [0, 1, 0], [-sy, 0, cy]])
    rz = np.array([[cz, -sz, 0], [sz, cz, 0], [0, 0, 1]])
    return rz @ rx @ ry, np.array(p[3:6])


def _matrix_by_angle(t, k):
    (cx, cy, cz), (sx, sy, sz) = np.cos(list(t.parameters)[:3]), np.sin(list(t.parameters)[:3])
    rx = np.array([[1, 0, 0], [0, cx, -sx], [0, sx, cx]])
    ry = np.array([[cy, 0, sy], [0, 1, 0], [-sy, 0, cy]])
    rz = np.array([[cz, -sz, 0], [sz, cz, 0], [0, 0, 1]])
    d = [np.array([[0, 0, 0], [0, -sx, -cx], [0, cx, -sx]]), np.array([[-sy, 0, cy], [0, 0, 0], [-cy, 0, -sy]]),
         np.array([[-sz, -cz, 0], [cz, -sz, 0], [0, 0, 0]])]
    return [rz @ d[0] @ ry, rz @ rx @ d[1], d[2] @ rx @ ry][k]


def _mi_exact(g, m, points, bins, binning, t, derivative):
    nb = binning.bins
    mat, trans = _matrix(t)
    p = points.t()
    q = torch.stack([float(mat[a, 0]) * p[0] + float(mat[a, 1]) * p[1] + float(mat[a, 2]) * p[2] + float(trans[a]) for a in range(3)])
    c = _index(g, q)
    v = _sample(m, c)
    keep = _inside(m, c) & (v >= binning.moving_min) & (v <= binning.moving_max)
    c, v, p, f = c[:, keep], v[keep], p[:, keep], bins[keep]
    term = (v - binning.moving_min) / binning.moving_bin_size + 2.0
    at = term.long().clamp(2, nb - 3)
    joint = torch.zeros(nb * nb, device="cuda", dtype=torch.float64)
    for k in range(-1, 3):
        joint.index_add_(0, f * nb + at + k, _bspline((at + k).double() - term))
    joint = joint.view(nb, nb) / joint.sum()
    fm = torch.bincount(f, minlength=nb).double() / f.numel()
    mm = joint.sum(0)
    ok = (fm[:, None] > EPS) & (mm[None, :] > EPS) & (joint > EPS)
    pr = torch.where(ok, torch.log(torch.where(ok, joint / mm[None, :], 1.0)), 0.0)
    lf = torch.log(torch.where(fm > EPS, fm, 1.0))
    value = -torch.where(ok, joint * (pr - lf[:, None]), 0.0).sum()
    if not derivative:
        return float(value)
    ratio = (-pr / (binning.moving_bin_size * f.numel())).reshape(-1)
    w = torch.zeros_like(term)
    for k in range(-1, 3):
        w += _bspline_d((at + k).double() - term) * ratio[f * nb + at + k]
    grad = []
    for a in range(3):
        up, down = c.clone(), c.clone()
        up[a] += 0.5
        down[a] -= 0.5
        d = (_sample(m, up) - _sample(m, down)) / float(g.spacing[a])
        grad.append(torch.where(_inside(m, up) & _inside(m, down), d, 0.0))
    if t.kind == 1:
        out = [(w * grad[r] * p[k]).sum() for r in range(3) for k in range(3)]
    else:
        out = []
        for k in range(3):
            d = _matrix_by_angle(t, k)
            out.append(sum((w * grad[r] * (float(d[r, 0]) * p[0] + float(d[r, 1]) * p[1] + float(d[r, 2]) * p[2])).sum() for r in range(3)))
    out += [(w * grad[r]).sum() for r in range(3)]
    return {"value": float(value), "derivative": np.array([float(x) for x in out])}


def _box(v, r):
    """Window sums of v over (2 r + 1) voxels an axis, clipped to the volume, added term by term."""
    for ax in (0, 1, 2):
        n = v.shape[ax]
        out = torch.zeros_like(v)
        for t in range(-r, r + 1):
            if abs(t) < n:
                lo, hi = max(0, -t), min(n, n - t)
                out.narrow(ax, lo, hi - lo).add_(v.narrow(ax, lo + t, hi - lo))
        v = out
    return v


def _gradients(v, g):
    """ITK's central differences along the physical axes: probes half a spacing away, zero where one leaves the volume."""
    x, y, z = _axes(g)
    c = torch.stack([x.expand(v.shape), y.expand(v.shape), z.expand(v.shape)])
    out = []
    d, s = g.dir_matrix(), list(g.spacing)
    for a in range(3):
        off = torch.tensor([d[a, k] * 0.5 * s[a] / s[k] for k in range(3)], device="cuda", dtype=torch.float64).view(3, 1, 1, 1)
        up, down = c + off, c - off
        out.append(torch.where(_inside(v, up) & _inside(v, down), (_sample(v, up) - _sample(v, down)) / s[a], 0.0))
    return out


def _cc_exact(case, seed):
    g, f, m = _cc_images(case, seed)
    r = case["radius"]
    n = _box(torch.ones_like(f), r)
    wf, wm = _box(f, r), _box(m, r)
    fbar, mbar = wf / n, wm / n
    sff = _box(f * f, r) - fbar * wf
    smm = _box(m * m, r) - mbar * wm
    sfm = _box(f * m, r) - fbar * wm
    product = sff * smm
    big = product.abs() > EPS
    value = -float(torch.where(big, sfm * sfm / torch.where(big, product, 1.0), 1.0).mean())
    ok = (sff > EPS) & (smm > EPS)
    k = torch.where(ok, 2 * sfm / torch.where(ok, product, 1.0), 0.0)
    fi, mi = f - fbar, m - mbar
    cf = k * (fi - torch.where(ok, sfm / torch.where(ok, smm, 1.0), 0.0) * mi)
    cm = k * (mi - torch.where(ok, sfm / torch.where(ok, sff, 1.0), 0.0) * fi)
    return [torch.stack([cf * d for d in _gradients(m, g)]), torch.stack([cm * d for d in _gradients(f, g)]),
            torch.tensor([value, value], dtype=torch.float64)]


def exact(case, seed):
    kind = case["kind"]
    if kind == "cc":
        return _cc_exact(case, seed)
    if kind.startswith("mi_"):
        g, m, points, bins, binning, ts = _level(case, seed)
        if kind == "mi_values":
            return np.array([_mi_exact(g, m, points, bins, binning, t, False) for t in ts])
        return _mi_exact(g, m, points, bins, binning, ts[0], kind == "mi_gradient")
    # whole stages and registrations: chains of hundreds of line searches, metrics and inversions
    # whose 64-bit form would be an engine of its own
    return None
