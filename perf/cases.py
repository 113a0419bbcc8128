"""The work that programs built on this package spend their time in, as measurable cases.

Every case goes through the public entry points (the autograd Functions and
modules of totrilib_amd.render, .reconstruct and .util).  Families:

  confocal    a step of a confocal fit: the render of an albedo volume, and the
              gradient of what the program makes of it with respect to the
              albedo (and the scan points, when they are calibrated too);
              float32, 16-bit transient storage, or float64
  backproject a reconstruction by VolumeRenderConfocal.apply_transposed
  velten      confocal Velten backprojection
  velten_ex   exhaustive (scan x laser) Velten backprojection
  arellano    ellipsoid backprojection of a thresholded capture
  exhaustive  exhaustive render and its albedo gradient
  splat       RBF splat and the RBF gradient, truncated or over the whole grid
  fk          f-k migration

listed() holds sizes of the benchmark, the tests and the small calls of a
fitting loop; draw() spreads over the same ranges.
"""
import math

import torch

from totrilib_amd.data.util import make_wall_grid
from totrilib_amd.reconstruct import (BackprojectionConfocalVelten,
                                      BackprojectionExhaustiveArellano,
                                      BackprojectionExhaustiveVelten, FkMigration)
from totrilib_amd.render.volume import VolumeRenderConfocal, VolumeRenderExhaustive
from totrilib_amd.types import BinDef, VolumeDef
from totrilib_amd.util import Rbf2VolumeGaussian

DEV = "cuda:0"
DTYPES = {"float32": torch.float32, "float64": torch.float64,
          "bfloat16": torch.bfloat16, "float16": torch.float16}


def listed():
    return [
        # One step of an interactive low-resolution fit: the smallest call in
        # use, where launches and host latency count as much as arithmetic.
        dict(name="confocal_small", family="confocal", X=32, Y=32, Z=32, scan="grid", nx=16, ny=16,
             T=256, albedo="dense", dtype="float32", storage="float32", grad="volume"),
        # The benchmark's step: 128^3 voxels, 64x64 wall grid, 1024 bins,
        # 3 % of the voxels occupied.
        dict(name="confocal_step", family="confocal", X=128, Y=128, Z=128, scan="grid", nx=64, ny=64,
             T=1024, albedo="sparse", dtype="float32", storage="float32", grad="volume"),
        # A fit to a real capture: galvo points off the ideal grid, odd sizes,
        # a hidden surface, and the scan points calibrated along with it.
        dict(name="confocal_capture", family="confocal", X=90, Y=84, Z=77, scan="jitter", nx=47, ny=41,
             T=601, albedo="surface", dtype="float32", storage="float32", grad="both"),
        # An off-grid capture in the middle of a solve: every voxel is nonzero.
        dict(name="confocal_dense", family="confocal", X=64, Y=64, Z=64, scan="jitter", nx=48, ny=48,
             T=512, albedo="dense", dtype="float32", storage="bfloat16", grad="volume"),
        # float64, as gradient checks and reference solutions run it.
        dict(name="confocal_f64", family="confocal", X=32, Y=32, Z=32, scan="grid", nx=16, ny=16,
             T=256, albedo="dense", dtype="float64", storage="float64", grad="volume"),
        # The large reconstruction at one GPU's share of its scan, 16-bit capture.
        dict(name="backproject_large", family="backproject", X=192, Y=192, Z=192, scan="grid",
             nx=128, ny=64, T=2048, storage="float16"),
        # Backprojections at the benchmark's sizes.
        dict(name="velten", family="velten", B=1, D=64, H=64, W=64, nx=32, ny=32, T=512, origin=False),
        dict(name="velten_exhaustive", family="velten_ex", B=1, D=64, H=64, W=64, nx=16, ny=16, nl=4,
             T=512, origin=True),
        dict(name="arellano", family="arellano", B=1, D=64, H=64, W=64, nx=16, ny=16, nl=4, T=512,
             filled=0.05),
        # The exhaustive render with its gradient, 5 % of the voxels occupied.
        dict(name="exhaustive_step", family="exhaustive", B=1, D=64, H=64, W=64, nx=16, ny=16, nl=4,
             T=512, filled=0.05),
        # The splat step of an RBF fit: over the whole grid (the default).
        dict(name="splat_full", family="splat", B=1, N=2000, A=1, D=64, H=80, W=96, truncation=0.0),
        # f-k migration of a 64x64 wall, 512 bins.
        dict(name="fk", family="fk", D=512, H=64, W=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["confocal", "confocal", "confocal", "backproject", "velten", "velten_ex",
                         "arellano", "exhaustive", "splat", "splat", "fk"])
    if family in ("confocal", "backproject"):
        scan = rng.choice(["grid", "jitter"])
        # half of the grids have the power-of-two sizes that programs prefer
        two = scan == "grid" and rng.random() < 0.5
        storage = rng.choice(["float32", "float32", "float32", "bfloat16", "float16"])
        dtype = "float32"
        if family == "confocal" and rng.random() < 0.2:
            dtype = storage = "float64"
        while True:
            dims = [2 ** rng.randint(4, 7) if two else _log_int(rng, 16, 144) for _ in range(3)]
            n = [2 * _log_int(rng, 4, 40) if two else _log_int(rng, 8, 80) for _ in range(2)]
            T = _log_int(rng, 128, 2048)
            cost = dims[0] * dims[1] * n[0] * n[1] * T
            if 1e6 < cost < (1e9 if dtype == "float64" else 7e10):
                break
        case = dict(family=family, X=dims[0], Y=dims[1], Z=dims[2], scan=scan, nx=n[0], ny=n[1], T=T,
                    storage=storage)
        if family == "confocal":
            case.update(albedo=rng.choice(["sparse", "dense", "surface"]), dtype=dtype,
                        grad="volume" if dtype == "float64" else rng.choice(["volume", "volume", "both"]))
        return case
    if family == "fk":
        if rng.random() < 0.6:
            return dict(family=family, D=2 ** rng.randint(6, 10), H=2 ** rng.randint(4, 6),
                        W=2 ** rng.randint(4, 6))
        return dict(family=family, D=_log_int(rng, 60, 1000), H=_log_int(rng, 16, 64),
                    W=_log_int(rng, 16, 64))
    if family == "splat":
        truncation = rng.choice([0.0, 0.0, 3.0, 3.5])
        while True:
            dims = [_log_int(rng, 16, 128) for _ in range(3)]
            N = _log_int(rng, 50, 20000)
            cost = N * dims[0] * dims[1] * dims[2]
            if truncation > 0 or cost < 5e9:
                break
        return dict(family=family, B=rng.choice([1, 1, 1, 2]), N=N, A=rng.choice([0, 1, 1, 1, 3]),
                    D=dims[0], H=dims[1], W=dims[2], truncation=truncation)
    while True:
        dims = [_log_int(rng, 16, 80) for _ in range(3)]
        n = [_log_int(rng, 8, 40) for _ in range(2)]
        nl = 0 if family == "velten" else _log_int(rng, 1, 6)
        T = _log_int(rng, 128, 1024)
        pairs = n[0] * n[1] * max(1, nl * nl)
        if pairs * dims[0] * dims[1] * dims[2] < 1.2e9 and pairs * T < 8e6:
            break
    case = dict(family=family, B=rng.choice([1, 1, 2]), D=dims[0], H=dims[1], W=dims[2], nx=n[0],
                ny=n[1], T=T)
    if family != "velten":
        case["nl"] = nl
    if family in ("velten", "velten_ex"):
        case["origin"] = rng.random() < 0.5
    else:
        case["filled"] = round(rng.uniform(0.02, 0.1), 3)
    return case


# ---------------------------------------------------------------------------
# geometry and inputs
# ---------------------------------------------------------------------------
BOX_START = (-1.0, -1.0, 0.5)
BOX_END = (1.0, 1.0, 2.5)
BOX_SIZE = (2.0, 2.0, 2.0)
LASER_Z = -1.0           # sensor and laser stand 1 m in front of the wall


def _rand(gen, *shape, dtype=torch.float32):
    return torch.rand(shape, generator=gen, device=DEV, dtype=dtype)


def _randn(gen, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=gen, device=DEV, dtype=dtype)


def _scan(case, gen):
    """[N, 3] wall points: the ideal grid, or a grid that a galvo hits 2 mm off."""
    p = make_wall_grid(x_res=case["nx"], y_res=case["ny"], device=DEV)
    if case["scan"] == "jitter":
        p = p + 0.002 * _randn(gen, *p.shape)
    return p


def _albedo(case, gen):
    X, Y, Z = case["X"], case["Y"], case["Z"]
    if case["albedo"] == "dense":        # an iterate of a nonnegative solve
        return _rand(gen, X, Y, Z) + 0.01
    if case["albedo"] == "sparse":       # 3 % of the voxels, anywhere
        return _rand(gen, X, Y, Z) * (_rand(gen, X, Y, Z) < 0.03)
    # a hidden surface: a smooth sheet, two voxels thick, over part of the columns
    x = torch.linspace(-1, 1, X, device=DEV)[:, None]
    y = torch.linspace(-1, 1, Y, device=DEV)[None, :]
    a = _rand(gen, 6)
    h = 0.5 + 0.2 * (a[0] - 0.5) * x + 0.2 * (a[1] - 0.5) * y \
        + 0.15 * torch.sin(3 * a[2] * x + 4 * a[3] * y)
    inside = ((x - 0.6 * (a[4] - 0.5)) ** 2 + (y - 0.6 * (a[5] - 0.5)) ** 2) < 0.45
    z = torch.arange(Z, device=DEV)[None, None, :]
    near = (z - (h * Z).floor()[:, :, None]).abs() < 1.5
    return (0.2 + 0.8 * _rand(gen, X, Y, Z)) * (near & (z >= (h * Z).floor()[:, :, None])) \
        * inside[:, :, None]


def _confocal_bins(case):
    """One-way bin width with which T bins reach the box's far corner."""
    far = math.sqrt(2.0 ** 2 + 2.0 ** 2 + 2.5 ** 2)
    return float(torch.tensor(far / case["T"], dtype=torch.float32))


def _capture(gen, *shape):
    """Photon histogram: dark counts, and returns that fall off along the bins."""
    base = 0.05 * _rand(gen, *shape)
    return base + _rand(gen, *shape) ** 4


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    f = case["family"]
    s = {"case": case}
    if f in ("confocal", "backproject"):
        dt = DTYPES[case.get("dtype", "float32")]
        s["points"] = _scan(case, gen).to(dt).T.contiguous()
        s["width"] = _confocal_bins(case)
        n, T = s["points"].shape[1], case["T"]
        if f == "confocal":
            s["volume"] = _albedo(case, gen).to(dt).contiguous().requires_grad_(True)
            if case["grad"] == "both":
                s["points"].requires_grad_(True)
            s["upstream"] = _randn(gen, n, T).to(DTYPES[case["storage"]])
        else:
            s["transient"] = _capture(gen, n, T).to(DTYPES[case["storage"]])
        return s
    if f == "splat":
        B, N, A = case["B"], case["N"], case["A"]
        s["def"] = VolumeDef(BOX_START, BOX_END, (case["D"], case["H"], case["W"]))
        lo, hi = _sigmas(case)
        sigma = lo + (hi - lo) * _rand(gen, B, N, 1)
        s["rbf"] = torch.cat([_rand(gen, B, N, 2) * 2 - 1, _rand(gen, B, N, 1) * 2 + 0.5, sigma,
                              _rand(gen, B, N, A)], 2).requires_grad_(True)
        s["upstream"] = _randn(gen, B, 1 + A, case["D"], case["H"], case["W"])
        return s
    if f == "fk":
        s["transient"] = _capture(gen, 1, case["D"], case["H"], case["W"])
        s["fk"] = FkMigration(*_fk_extent(case))
        return s
    # wall points of the volume backprojections and the exhaustive render
    B, T = case["B"], case["T"]
    s["def"] = VolumeDef(BOX_START, BOX_END, (case["D"], case["H"], case["W"]))
    scan = make_wall_grid(x_res=case["nx"], y_res=case["ny"], device=DEV).expand(B, -1, 3)
    scan = scan + 0.002 * _randn(gen, *scan.shape)
    s["scan"] = scan.contiguous()
    S = scan.shape[1]
    far = 2 * math.sqrt(2.0 ** 2 + 2.0 ** 2 + 2.5 ** 2)
    offset = 0.0
    origin = None
    if case.get("origin"):
        origin = torch.tensor([0.1, -0.2, LASER_Z], device=DEV).expand(B, 3).contiguous()
        far, offset = far + 2.0, 2.0
    s["scan_origin"] = origin
    s["bins"] = BinDef((far - offset) / T, offset, T)
    if f == "velten":
        s["transient"] = _capture(gen, B, T, S)
        return s
    laser = make_wall_grid(-0.5, 0.5, case["nl"], -0.5, 0.5, case["nl"], device=DEV).expand(B, -1, 3)
    laser = laser + 0.002 * _randn(gen, *laser.shape)
    s["laser"] = laser.contiguous()
    s["laser_origin"] = origin
    L = laser.shape[1]
    if f in ("arellano", "exhaustive"):       # these take [B, 3, N] points
        s["scan"] = s["scan"].transpose(1, 2).contiguous()
        s["laser"] = s["laser"].transpose(1, 2).contiguous()
    if f == "exhaustive":
        shape = (B, case["D"], case["H"], case["W"])
        s["volume"] = (_rand(gen, *shape) * (_rand(gen, *shape) < case["filled"])).requires_grad_(True)
        s["upstream"] = _randn(gen, B, T, S, L)
        return s
    s["transient"] = _capture(gen, B, T, S, L)
    if f == "arellano":
        s["transient"] = s["transient"] * (_rand(gen, B, T, S, L) < case["filled"])
    return s


def _sigmas(case):
    """Fits cut off many small blobs, and let a few wide ones reach everywhere."""
    return (0.01, 0.05) if case["truncation"] > 0 else (0.03, 0.1)


def _fk_extent(case):
    return (case["D"] * 0.0025, 2.0, 2.0)


def run(state):
    case = state["case"]
    f = case["family"]
    if f == "confocal":
        storage = DTYPES[case["storage"]]
        tr = VolumeRenderConfocal.apply(state["volume"], state["points"], BOX_START, BOX_SIZE, case["T"],
                                        state["width"], 0.0, storage)
        wrt = [state["volume"]] + ([state["points"]] if case["grad"] == "both" else [])
        return [tr.detach(), *torch.autograd.grad(tr, wrt, state["upstream"])]
    if f == "backproject":
        return VolumeRenderConfocal.apply_transposed(
            state["transient"], state["points"], BOX_START, BOX_SIZE, (case["X"], case["Y"], case["Z"]),
            state["width"], 0.0)
    if f == "velten":
        return BackprojectionConfocalVelten.apply(state["transient"], state["scan"], state["def"],
                                                  state["bins"], state["scan_origin"])
    if f == "velten_ex":
        return BackprojectionExhaustiveVelten.apply(
            state["transient"], state["scan"], state["laser"], state["def"], state["bins"],
            state["scan_origin"], state["laser_origin"])
    if f == "arellano":
        return BackprojectionExhaustiveArellano.apply(state["transient"], state["scan"], state["laser"],
                                                      state["def"], state["bins"])
    if f == "exhaustive":
        tr = VolumeRenderExhaustive.apply(state["volume"], state["scan"], state["laser"], state["def"],
                                          state["bins"])
        return [tr.detach(), *torch.autograd.grad(tr, state["volume"], state["upstream"])]
    if f == "splat":
        v = Rbf2VolumeGaussian.apply(state["rbf"], state["def"], case["truncation"])
        return [v.detach(), *torch.autograd.grad(v, state["rbf"], state["upstream"])]
    return state["fk"](state["transient"])


def _samples(case):
    """About how many (scan point, column, bin) samples lie in the box: a
    column's bins span the box's depth."""
    depth = 2.0 / _confocal_bins(case)
    return case["X"] * case["Y"] * case["nx"] * case["ny"] * min(case["T"], 0.65 * depth)


def work(case):
    """Inputs read once, outputs written once, and the operations of the
    formulas: 18 a render sample, 20 an adjoint sample, 30 a scan-point
    gradient sample, 14 a voxel-scan pair, and so on."""
    f = case["family"]
    if f in ("confocal", "backproject"):
        V, NT = case["X"] * case["Y"] * case["Z"], case["nx"] * case["ny"] * case["T"]
        size = {"float32": 4, "float64": 8}.get(case["storage"], 2)
        vsize = 8 if case.get("dtype") == "float64" else 4
        n = _samples(case)
        if f == "backproject":
            return {"bytes": vsize * V + size * NT, "flops": 20 * n}
        both = case["grad"] == "both"
        return {"bytes": 2 * vsize * V + 2 * size * NT, "flops": (38 + (30 if both else 0)) * n}
    if f == "fk":
        n = case["D"] * case["H"] * case["W"]
        return {"bytes": 8 * n, "flops": 2 * n * (10 * math.log2(2 * n) + 80)}
    if f == "splat":
        V = case["D"] * case["H"] * case["W"]
        pairs = case["B"] * case["N"] * V
        if case["truncation"] > 0:
            # mean of (k sigma)^3 for a uniform sigma, in units of the 8 m^3 box
            lo, hi = _sigmas(case)
            cube = (hi ** 4 - lo ** 4) / (4 * (hi - lo))
            pairs *= min(1.0, 4.19 * case["truncation"] ** 3 * cube / 8.0)
        return {"bytes": 4 * case["B"] * (2 * (1 + case["A"]) * V + 2 * (4 + case["A"]) * case["N"]),
                "flops": 39 * pairs}
    V = case["B"] * case["D"] * case["H"] * case["W"]
    pairs = case["nx"] * case["ny"] * max(1, case.get("nl", 0) ** 2)
    data = case["B"] * pairs * case["T"]
    flops = {"velten": 14 * V * pairs, "velten_ex": 8 * V * pairs,
             "arellano": 30 * V / case["D"] * pairs * case["T"] * case.get("filled", 0),
             "exhaustive": 40 * V * pairs * (1 + case.get("filled", 0))}[f]
    both = 2 if f == "exhaustive" else 1
    return {"bytes": 4 * both * (V + data), "flops": flops}


# ---------------------------------------------------------------------------
# the same results in 64 bits, from the formulas
# ---------------------------------------------------------------------------
def _centres(start, size, n):
    return start + (torch.arange(n, device=DEV, dtype=torch.float64) + 0.5) * size / n


def _exact_confocal(case, s):
    X, Y, Z, T = case["X"], case["Y"], case["Z"], case["T"]
    pts = s["points"].detach().double()
    N = pts.shape[1]
    if X * Y * N * T > 2.5e10:
        return None
    forward = case["family"] == "confocal"
    both = forward and case["grad"] == "both"
    G = (s["upstream"] if forward else s["transient"]).double()
    if case.get("dtype") == "float64":    # float64 renders keep a float32 bin radius
        tc = (torch.arange(T, device=DEV, dtype=torch.float32) * s["width"]).double()
    else:
        tc = torch.arange(T, device=DEV, dtype=torch.float64) * s["width"]
    x = _centres(BOX_START[0], BOX_SIZE[0], X)
    y = _centres(BOX_START[1], BOX_SIZE[1], Y)
    scale = Z / BOX_SIZE[2]
    C = X * Y
    base = (torch.arange(C, device=DEV) * Z)[:, None]
    vol = s["volume"].detach().double().reshape(-1) if forward else None
    render = torch.zeros(N, T, device=DEV, dtype=torch.float64)
    grad = torch.zeros(C * Z, device=DEV, dtype=torch.float64)
    gpts = torch.zeros(3, N, device=DEV, dtype=torch.float64)
    t4 = torch.where(tc > 0, tc, torch.ones_like(tc)) ** -8
    for i in range(N):
        dx = (pts[0, i] - x)[:, None].expand(X, Y).reshape(-1, 1)
        dy = (pts[1, i] - y)[None, :].expand(X, Y).reshape(-1, 1)
        d2 = (tc * tc)[None, :] - dx * dx - dy * dy
        depth = d2.clamp(min=0).sqrt()
        zh = (pts[2, i] + depth - BOX_START[2]) * scale - 0.5
        zi = zh.floor()
        live = (d2 > 0) & (zi >= 0) & (zi + 1 < Z)
        a = zh - zi
        f2 = torch.where(live, d2 * d2 * t4, torch.zeros_like(d2))
        at = (zi.clamp(0, max(Z - 2, 0)).long() + base)
        if forward:
            v0, v1 = vol[at], vol[at + 1]
            f1 = (1 - a) * v0 + a * v1
            render[i] = (f1 * f2).sum(0)
            if both:
                g = G[i][None, :]
                inv = torch.where(live, 1 / depth.clamp(min=1e-300), torch.zeros_like(depth))
                slope = scale * (v1 - v0) * f2
                h = -(4 * f1 * torch.where(live, d2 * t4, torch.zeros_like(d2)) + slope * inv) * g
                gpts[0, i], gpts[1, i] = (h * dx).sum(), (h * dy).sum()
                gpts[2, i] = (slope * g).sum()
        w = f2 * G[i][None, :]
        grad.index_add_(0, at.reshape(-1), ((1 - a) * w).reshape(-1))
        grad.index_add_(0, (at + 1).reshape(-1), (a * w).reshape(-1))
    grad = grad.view(X, Y, Z)
    if not forward:
        return grad
    return [render, grad, gpts] if both else [render, grad]


def _grid(case, s):
    """Voxel positions of the inclusive grid, [D * H * W, 3] in float64."""
    axes = [torch.linspace(a, b, n, device=DEV, dtype=torch.float64) if n > 1 else
            torch.full((1,), a, device=DEV, dtype=torch.float64)
            for a, b, n in zip(BOX_START, BOX_END, (case["W"], case["H"], case["D"]))]
    z, y, x = torch.meshgrid(axes[2], axes[1], axes[0], indexing="ij")
    return torch.stack([x.reshape(-1), y.reshape(-1), z.reshape(-1)], 1)


def _dist(q, p):
    return (q - p).square().sum(-1).sqrt()


def _exact_velten(case, s):
    bins, T = s["bins"], case["T"]
    q = _grid(case, s)
    out = torch.zeros(case["B"], q.shape[0], device=DEV, dtype=torch.float64)
    ex = case["family"] == "velten_ex"
    for b in range(case["B"]):
        scan = s["scan"][b].double()
        so = torch.zeros(scan.shape[0], device=DEV, dtype=torch.float64)
        if s["scan_origin"] is not None:
            so = _dist(scan, s["scan_origin"][b].double())
        tr = s["transient"][b].double()
        dl = None
        if ex:
            laser = s["laser"][b].double()
            dl = torch.stack([_dist(q, laser[k]) for k in range(laser.shape[0])], 1)
            if s["laser_origin"] is not None:
                dl = dl + _dist(laser, s["laser_origin"][b].double())
        for i in range(scan.shape[0]):
            d = (so[i] + _dist(q, scan[i]))[:, None]
            d = d + dl if ex else 2 * d
            t = ((d - bins.offset) / bins.width + 0.5).floor().long()
            row = tr[:, i] if ex else tr[:, i, None]
            v = row.gather(0, t.clamp(0, T - 1))
            out[b] += torch.where((t >= 0) & (t < T), v, torch.zeros_like(v)).sum(1)
    return out.view(case["B"], case["D"], case["H"], case["W"])


def _exact_arellano(case, s):
    bins, D = s["bins"], case["D"]
    HW = case["H"] * case["W"]
    col = _grid(case, s)[:HW]
    start, end = col, col + torch.tensor([0.0, 0.0, BOX_END[2] - BOX_START[2]], device=DEV,
                                         dtype=torch.float64)
    out = torch.zeros(case["B"], D, HW, device=DEV, dtype=torch.float64)
    for b in range(case["B"]):
        scan, laser = s["scan"][b].double().T, s["laser"][b].double().T
        for i in range(scan.shape[0]):
            for k in range(laser.shape[0]):
                tr = s["transient"][b, :, i, k].double()
                t = tr.nonzero()[:, 0]
                tc = t * bins.width + bins.offset
                n = scan[i] - laser[k]
                ln = n.norm()
                n = n / ln if ln > 1e-6 else n
                keep = tc > ln
                val, tc = tr[t][keep][:, None], tc[keep][:, None]
                c = 0.5 * (scan[i] + laser[k])
                r1 = (tc * tc / 4 - ln * ln / 4).sqrt()
                sc = (r1 / (tc / 2) - 1)[..., None]
                a = (start - c)[None] + sc * ((start - c) @ n)[None, :, None] * n
                e = (end - c)[None] + sc * ((end - c) @ n)[None, :, None] * n
                d = e - a
                rl = d.norm(dim=-1)
                d = d / rl[..., None]
                v0 = (d * a).sum(-1)
                v1 = v0 * v0 - ((a * a).sum(-1) - r1 * r1)
                hit = v1 > 0
                v1 = v1.clamp(min=0).sqrt()
                r = torch.where(-v0 - v1 < 0, -v0 + v1, -v0 - v1)
                z = (r / rl * D + 0.5).trunc()
                hit = hit & (z >= 0) & (z < D)
                at = z.clamp(0, D - 1).long() * HW + torch.arange(HW, device=DEV)[None, :]
                out[b].view(-1).index_add_(0, at.reshape(-1),
                                           torch.where(hit, val, torch.zeros_like(r)).reshape(-1))
    return out.view(case["B"], D, case["H"], case["W"])


def _exact_exhaustive(case, s):
    bins, T = s["bins"], case["T"]
    D, H, W = case["D"], case["H"], case["W"]
    z = _centres(BOX_START[2], BOX_SIZE[2], D)
    y = _centres(BOX_START[1], BOX_SIZE[1], H)
    x = _centres(BOX_START[0], BOX_SIZE[0], W)
    zz, yy, xx = (v.reshape(-1) for v in torch.meshgrid(z, y, x, indexing="ij"))
    h = torch.tensor([0.0, 0.0, 0.5 * BOX_SIZE[2] / D], device=DEV, dtype=torch.float64)
    q = torch.stack([xx, yy, zz], 1)
    vol, G = s["volume"].detach().double(), s["upstream"].double()
    render, grad = torch.zeros_like(G), torch.zeros(case["B"], D * H * W, device=DEV, dtype=torch.float64)
    for b in range(case["B"]):
        occ = vol[b].reshape(-1)
        full = occ.nonzero()[:, 0]
        scan, laser = s["scan"][b].double().T, s["laser"][b].double().T
        near = [(_dist(q - h, p), _dist(q + h, p)) for p in laser]
        for i in range(scan.shape[0]):
            n0, n1 = _dist(q - h, scan[i]), _dist(q + h, scan[i])
            for k in range(laser.shape[0]):
                d0, d1 = n0 + near[k][0], n1 + near[k][1]
                b0 = (torch.minimum(d0, d1) - bins.offset) / bins.width
                b1 = (torch.maximum(d0, d1) - bins.offset) / bins.width
                span = b1 - b0
                f, l = b0.floor().long(), b1.floor().long()
                ok = (l >= 0) & (f < T)
                b0, f = torch.where(f < 0, torch.zeros_like(b0), b0), f.clamp(min=0)
                b1, l = torch.where(l >= T, torch.full_like(b1, T - 1), b1), l.clamp(max=T - 1)
                frac = torch.where(ok, 1 / span, torch.zeros_like(span))
                one = f == l
                for j in range(int((l - f)[ok].max()) + 1 if bool(ok.any()) else 0):
                    t = f + j
                    w = torch.where(t == l, (b1 - l) * frac, frac)
                    if j == 0:
                        w = torch.where(one, ok.double(), (1 - (b0 - f)) * frac)
                    w = torch.where(ok & (t <= l), w, torch.zeros_like(w))
                    t = t.clamp(0, T - 1)
                    grad[b] += w * G[b, :, i, k][t]
                    render[b, :, i, k].index_add_(0, t[full], (w * occ)[full])
    return [render, grad.view(case["B"], D, H, W)]


def _exact_splat(case, s):
    B, N, A = case["B"], case["N"], case["A"]
    D, H, W = case["D"], case["H"], case["W"]
    if case["truncation"] == 0 and B * N * D * H * W > 6e9:
        return None
    axes = [torch.linspace(a, b, n, device=DEV, dtype=torch.float64)
            for a, b, n in zip(BOX_START, BOX_END, (W, H, D))]
    rbf, G = s["rbf"].detach().double(), s["upstream"].double()
    out = torch.zeros(B, 1 + A, D * H * W, device=DEV, dtype=torch.float64)
    grad = torch.zeros_like(rbf)
    step = [(b - a) / (n - 1) for a, b, n in zip(BOX_START, BOX_END, (W, H, D))]
    if case["truncation"] > 0:            # a window that holds the widest RBF
        reach = [min(n, 2 * int(case["truncation"] * 1.001 * _sigmas(case)[1] / d) + 4)
                 for n, d in zip((W, H, D), step)]
    else:
        reach = [W, H, D]
    chunk = max(1, int(2e7 / (reach[0] * reach[1] * reach[2])))

    def windows(r):
        """Flat voxel indices [n, K], offsets and Gaussians of a chunk's windows."""
        at, off = [], []
        for ax in range(3):
            lo = ((r[:, ax] - BOX_START[ax]) / step[ax]).round().long() - reach[ax] // 2
            lo = lo.clamp(min=0).clamp(max=axes[ax].shape[0] - reach[ax])
            k = lo[:, None] + torch.arange(reach[ax], device=DEV)
            at.append(k)
            off.append(r[:, ax, None] - axes[ax][k])
        n = r.shape[0]
        flat = (at[2][:, :, None, None] * H + at[1][:, None, :, None]) * W + at[0][:, None, None, :]
        dz, dy, dx = off[2][:, :, None, None], off[1][:, None, :, None], off[0][:, None, None, :]
        r2 = dx * dx + dy * dy + dz * dz
        sg = r[:, 3, None, None, None]
        g = torch.exp(-0.5 * r2 / (sg * sg))
        if case["truncation"] > 0:
            g = torch.where(r2 <= (case["truncation"] * sg) ** 2, g, torch.zeros_like(g))
        return flat.reshape(n, -1), (dx, dy, dz, r2), g

    for b in range(B):
        for c in range(0, N, chunk):
            r = rbf[b, c:c + chunk]
            flat, _, g = windows(r)
            g = g.reshape(r.shape[0], -1)
            if case["truncation"] == 0:
                out[b, 0] += g.sum(0)
                for a in range(A):
                    out[b, 1 + a] += r[:, 4 + a] @ g
            else:
                out[b, 0].index_add_(0, flat.reshape(-1), g.reshape(-1))
                for a in range(A):
                    out[b, 1 + a].index_add_(0, flat.reshape(-1), (g * r[:, 4 + a, None]).reshape(-1))
        norm = torch.where(out[b, 0] < 1e-8, torch.ones_like(out[b, 0]), out[b, 0])
        out[b, 1:] /= norm
        up = G[b].reshape(1 + A, -1)
        per = up[1:] / norm
        head = up[0] - (per * out[b, 1:]).sum(0)
        for c in range(0, N, chunk):
            r = rbf[b, c:c + chunk]
            n = r.shape[0]
            flat, (dx, dy, dz, r2), g = windows(r)
            u = head[flat].view_as(g)
            for a in range(A):
                pa = per[a][flat].view_as(g)
                grad[b, c:c + n, 4 + a] = (pa * g).sum((1, 2, 3))
                u = u + pa * r[:, 4 + a, None, None, None]
            m, sg = u * g, r[:, 3]
            for ax, d in enumerate((dx, dy, dz)):
                grad[b, c:c + n, ax] = -(m * d).sum((1, 2, 3)) / sg ** 2
            grad[b, c:c + n, 3] = (m * r2).sum((1, 2, 3)) / sg ** 3
    return [out.view(B, 1 + A, D, H, W), grad]


def _exact_fk(case, s):
    D, H, W = case["D"], case["H"], case["W"]
    depth, height, width = _fk_extent(case)
    f64 = dict(device=DEV, dtype=torch.float64)
    t = s["transient"][0].double().sqrt() * torch.linspace(0, 1, D, **f64)[:, None, None]
    t = torch.cat((t, torch.zeros_like(t)), 0)
    F = torch.fft.fftshift(torch.fft.fftn(t))
    x = torch.linspace(-1, 1, W, **f64).view(1, 1, W).expand(2 * D, H, W)
    y = torch.linspace(-1, 1, H, **f64).view(1, H, 1).expand(2 * D, H, W)
    z = torch.linspace(-1, 1, 2 * D, **f64).view(2 * D, 1, 1).expand(2 * D, H, W)
    zz = torch.sqrt((x * (W * depth) / (2 * D * width)) ** 2
                    + (y * (H * depth) / (2 * D * height)) ** 2 + z * z)
    grid = torch.stack((x, y, zz), 3)[None].expand(2, -1, -1, -1, -1)
    parts = torch.nn.functional.grid_sample(torch.stack((F.real, F.imag))[:, None], grid,
                                            align_corners=False)[:, 0]
    F = torch.complex(parts[0], parts[1]) * ((z > 0) * z.abs() / zz.clamp(min=1e-6))
    return torch.fft.ifftn(torch.fft.ifftshift(F)).abs()[None, :D]


def exact(case, seed):
    s = prepare(case, seed)
    f = case["family"]
    return {"confocal": _exact_confocal, "backproject": _exact_confocal, "velten": _exact_velten,
            "velten_ex": _exact_velten, "arellano": _exact_arellano, "exhaustive": _exact_exhaustive,
            "splat": _exact_splat, "fk": _exact_fk}[f](case, s)
