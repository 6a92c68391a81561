"""The calls a program makes of this library, as timed workloads.

Each case is one pass through the public entry points (`robartsvtk_amd.abi`,
`robartsvtk_amd.autograd`): rendering one view with every caster, loading a
new volume frame, rendering many poses, and the two gradient directions
(poses and volume).  `listed()` names them, `draw()` takes more of the same
ranges, `prepare()` makes what a program holds before the call, `run()` is
the call, and `exact()` gives the float results in 64 bits by plain torch.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from robartsvtk_amd import abi
from robartsvtk_amd.autograd import DrrRenderer, drr_render

SID, SOD, FOV = 1000.0, 600.0, 409.6  # C-arm geometry, mm


def listed():
    return [
        # One small projection: the preview of a 2D/3D registration, or one
        # evaluation of its cost function.  Launch and ray latency count.
        dict(name="drr_preview", kind="drr", nx=128, ny=128, nz=128, sx=2.0, sy=2.0, sz=2.0, w=128, h=128, step=1.0,
             skip=True, output="exp"),
        # The headline radiograph: 256^3 CT, one 1024^2 detector.
        dict(name="drr_frame", kind="drr", nx=256, ny=256, nz=256, sx=1.0, sy=1.0, sz=1.0, w=1024, h=1024, step=0.5,
             skip=True, output="exp"),
        # Interactive 1D transfer-function view of an 8-bit volume.
        dict(name="tf1d_view", kind="tf1d", nx=128, ny=128, nz=128, sx=1.0, sy=1.0, sz=1.0, w=512, h=512, step=0.5,
             dtype="u8", n=256, shaded=False, live=False),
        # Live 4D rendering: a new CT frame is loaded and shown, shaded, at
        # the mapper's own step and termination; ragged sizes.
        dict(name="tf1d_live_frame", kind="tf1d", nx=250, ny=250, nz=181, sx=0.9, sy=0.9, sz=1.2, w=800, h=600,
             step=1.0, dtype="i16", n=512, shaded=True, live=True),
        # 2D transfer function over value and precomputed gradient magnitude,
        # full HD.
        dict(name="tf2d_gradmag", kind="tf2d", nx=512, ny=512, nz=512, sx=1.0, sy=1.0, sz=1.0, w=1920, h=1080,
             step=0.5, n=256, gradmag=True, post=False),
        # The 2D mapper's own render: gradient per sample, shading, depth
        # outputs and the cel/distance pass; odd volume sizes.
        dict(name="tf2d_shaded", kind="tf2d", nx=301, ny=257, nz=180, sx=0.8, sy=0.8, sz=1.5, w=1280, h=720, step=1.0,
             n=256, gradmag=False, post=True),
        # In/Ex logic with the black keyhole.
        dict(name="inex_keyhole", kind="inex", nx=256, ny=256, nz=200, sx=1.0, sy=1.0, sz=1.25, w=640, h=480, step=1.0,
             n=256, keyhole=True),
        # Dual-energy pair of images.
        dict(name="dual_view", kind="dual", nx=320, ny=320, nz=211, sx=0.8, sy=0.8, sz=1.0, w=1024, h=768, step=1.0,
             n=256),
        # Biplane registration iteration, recorded once and replayed.
        dict(name="register_biplane", kind="register", nx=200, ny=200, nz=160, sx=1.2, sy=1.2, sz=1.5, views=2, w=200,
             h=180, step=1.0, captured=True),
        # Many-view registration iteration.
        dict(name="register_views", kind="register", nx=256, ny=256, nz=256, sx=1.0, sy=1.0, sz=1.0, views=16, w=512,
             h=512, step=0.5, captured=False),
        # One reconstruction iteration: the volume changed, so it is loaded,
        # rendered, and the gradients go back to volume and poses.
        dict(name="reconstruct", kind="reconstruct", nx=256, ny=256, nz=256, sx=1.0, sy=1.0, sz=1.0, views=16, w=512,
             h=512, step=0.5),
        # Many poses on detectors of different sizes: forward and pose
        # gradient for a loss of the program's own.
        dict(name="pose_batch", kind="poses", nx=512, ny=512, nz=400, sx=1.0, sy=1.0, sz=1.0, views=64, w=1024, h=1024,
             step=0.5),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["drr", "drr", "tf1d", "tf1d", "tf2d", "tf2d", "inex", "dual", "register", "register",
                       "reconstruct", "poses"])
    nx, ny, nz = (_log_int(rng, 64, 400) for _ in range(3))
    base = 230.0 / max(nx, ny)
    c = dict(kind=kind, nx=nx, ny=ny, nz=nz, sx=round(base * rng.uniform(0.8, 1.2), 3),
             sy=round(base * rng.uniform(0.8, 1.2), 3), sz=round(min(3.0 * base, 230.0 / nz) * rng.uniform(0.8, 1.2), 3),
             w=_log_int(rng, 96, 1400), h=_log_int(rng, 96, 1100), step=rng.choice([0.5, 0.75, 1.0, 1.0]))
    if kind == "drr":
        c.update(skip=rng.choice([True, True, False]), output=rng.choice(["exp", "L", "rgba"]))
    elif kind == "tf1d":
        c.update(dtype=rng.choice(["u8", "i16", "u16", "f32"]), n=rng.choice([256, 512, 1024]),
                 shaded=rng.choice([True, False]), live=rng.choice([True, False]))
    elif kind == "tf2d":
        c.update(n=rng.choice([128, 256, 512]), gradmag=rng.choice([True, False]), post=rng.choice([True, False]))
    elif kind == "inex":
        c.update(n=rng.choice([128, 256, 512]), keyhole=rng.choice([True, False]))
    elif kind == "dual":
        c.update(n=rng.choice([128, 256, 512]))
    else:
        views = _log_int(rng, 1, 24)
        c.update(views=views, w=_log_int(rng, 64, 560), h=_log_int(rng, 64, 560))
        if kind == "register":
            c.update(captured=rng.choice([True, False]))
    return c


# ---------------------------------------------------------------------------
# inputs
def _np_rng(case, seed, tag):
    return np.random.default_rng([int(seed) & 0x7FFFFFFF, tag, case["nx"], case["w"]])


def _spacing(case):
    return (float(case["sx"]), float(case["sy"]), float(case["sz"]))


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed((int(seed) & 0x7FFFFFFF) + 17)


def _axes(case):
    n = (case["nx"], case["ny"], case["nz"])
    x, y, z = (torch.arange(k, device="cuda", dtype=torch.float32) for k in n)
    return x[None, None, :], y[None, :, None], z[:, None, None]


def _ct(case, seed):
    """CT of a body in air, Hounsfield units as int16: soft tissue with
    scanner noise, bones, air at -1000."""
    r = _np_rng(case, seed, 1)
    x, y, z = _axes(case)
    n = np.array([case["nx"], case["ny"], case["nz"]], float)
    c = n * (0.5 + r.uniform(-0.02, 0.02, 3))
    body = n * [r.uniform(0.36, 0.42), r.uniform(0.26, 0.34), r.uniform(0.38, 0.44)]

    def inside(ctr, rad):
        q = ((x - ctr[0]) / rad[0]) ** 2 + ((y - ctr[1]) / rad[1]) ** 2 + ((z - ctr[2]) / rad[2]) ** 2
        return q <= 1.0

    hu = torch.empty((case["nz"], case["ny"], case["nx"]), device="cuda")
    hu.normal_(40.0, 20.0, generator=_gen(seed))
    for _ in range(6):
        hu.masked_fill_(inside(c + r.uniform(-0.55, 0.55, 3) * body, n * r.uniform(0.04, 0.12, 3)),
                        float(r.uniform(400.0, 1500.0)))
    hu.masked_fill_(~inside(c, body), -1000.0)
    return hu.round_().to(torch.int16)


def _blobs(case, seed, vmax, noise, detail):
    """Smooth blobs with sensor noise and (detail) several octaves of smooth
    structure, scaled to [0, vmax]."""
    r = _np_rng(case, seed, 2)
    x, y, z = _axes(case)
    n = np.array([case["nx"], case["ny"], case["nz"]], float)
    v = torch.zeros((case["nz"], case["ny"], case["nx"]), device="cuda")
    for _ in range(8):
        ctr, sig = n * r.uniform(0.2, 0.8, 3), n.min() * r.uniform(0.05, 0.16)
        amp = r.uniform(0.35, 1.0)
        ex, ey, ez = (torch.exp(-((a - float(k)) ** 2) / float(2 * sig * sig)) for a, k in zip((x, y, z), ctr))
        v.addcmul_(ez * ey, ex, value=float(amp))
    g = _gen(seed)
    if detail:
        amp, cells = 0.3, 10
        for _ in range(4):
            k = [max(2, round(cells * d / n.max())) for d in n[::-1]]
            grid = torch.randn((1, 1, *k), device="cuda", generator=g)
            v.add_(torch.nn.functional.interpolate(grid, size=v.shape, mode="trilinear", align_corners=True)[0, 0],
                   alpha=0.5 * amp)
            amp, cells = 0.5 * amp, 2 * cells
    lo, hi = (float(q) for q in torch.aminmax(v))
    v.sub_(lo).mul_(vmax / (hi - lo) if hi > lo else 0.0)
    if noise:
        v.add_(torch.rand(v.shape, device="cuda", generator=g), alpha=noise)
    return v.clamp_(0.0, vmax)


def _mu(hu):
    return (0.02 * (1.0 + hu.float() / 1000.0)).clamp_(min=0.0)


def _center(case):
    return np.array([(n - 1) * s * 0.5 for n, s in zip((case["nx"], case["ny"], case["nz"]), _spacing(case))])


def _cam(position, focal, up, angle, near, far):
    return dict(position=np.asarray(position, float), focal=np.asarray(focal, float), up=np.asarray(up, float),
                angle=float(angle), near=float(near), far=float(far))


def _extent(case):
    s = _spacing(case)
    return 0.5 * math.sqrt(sum((n * k) ** 2 for n, k in zip((case["nx"], case["ny"], case["nz"]), s))) + 4.0


def _drr_cam(case, angle):
    c, half = _center(case), _extent(case)
    d = np.array([math.cos(angle), math.sin(angle), 0.0])
    return _cam(c + SOD * d, c, (0, 0, 1), 2.0 * math.degrees(math.atan(0.5 * FOV / SID)), max(1.0, SOD - half),
                SOD + half)


def _scene_cam(case, seed):
    """An eye around the volume that frames it."""
    r = _np_rng(case, seed, 3)
    c, half = _center(case), _extent(case)
    z = r.uniform(-0.8, 0.8)
    a = r.uniform(0.0, 2.0 * math.pi)
    q = math.sqrt(1.0 - z * z)
    d = np.array([q * math.cos(a), q * math.sin(a), z])
    dist = 2.6 * half
    return _cam(c + dist * d, c, (0, 0, 1), 30.0, max(1e-3, dist - half), dist + half)


def _abi_cam(c):
    return abi.camera(c["position"], c["focal"], c["up"], c["angle"], (c["near"], c["far"]))


def _poses(case, seed):
    """Cameras, detector sizes and rigid poses of a multi-view case."""
    r = _np_rng(case, seed, 4)
    n = case["views"]
    if case["kind"] == "poses":  # one C-arm position, many candidate poses, detectors of 1/4 to the full size
        cams = [_drr_cam(case, 0.0)] * n
        f = [0.25 * (1 + (5 * i + 3 * (i // 4)) % 4) for i in range(n)]
        sizes = [(max(16, round(case["w"] * k)), max(16, round(case["h"] * k))) for k in f]
        rot, tr = 10.0, 20.0
    else:
        cams = [_drr_cam(case, math.pi * i / n) for i in range(n)]
        sizes = [(case["w"], case["h"])] * n
        rot, tr = 5.0, 10.0
    p = np.concatenate([np.radians(r.uniform(-rot, rot, (n, 3))), r.uniform(-tr, tr, (n, 3))], 1)
    return cams, sizes, p


def _march(case, term):
    return abi.MarchParams(float(case["step"]), float(term), 1, int(case.get("skip", True)), 1)


def _drr_params(case):
    d = abi.DrrParams()
    if case["kind"] in ("register", "reconstruct"):  # volumes of attenuation
        d.ct_intercept, d.ct_slope = 0.0, 1.0
    else:  # Hounsfield units
        d.ct_intercept, d.ct_slope = 0.02, 2e-5
    d.ct_offset = 1.0
    d.output = {"exp": abi.DRR_F32_EXP_NEG_L, "L": abi.DRR_F32_L, "rgba": abi.DRR_RGBA8_REF}[case.get("output", "exp")]
    d.tint[:] = [255, 240, 220, 200]
    return d


def _curve(xs, ys, lo, hi, n):
    return np.interp(lo + np.arange(n) * ((hi - lo) / (n - 1)), xs, ys).astype(np.float32)


def _tf1d(case, seed, ctx, lo, hi):
    r = _np_rng(case, seed, 5)
    n, w = case["n"], hi - lo
    xs = [lo, lo + r.uniform(0.2, 0.25) * w, lo + r.uniform(0.5, 0.6) * w, hi]
    alpha = _curve(xs, [0.0, 0.0, r.uniform(0.05, 0.1), r.uniform(0.4, 0.6)], lo, hi, n)
    rgb = np.stack([_curve(xs, r.uniform(0, 1, 4), lo, hi, n) for _ in range(3)], 1)
    if case["shaded"]:
        ga = _curve([0.0, 0.02, 0.2, 1.0], [0.2, 0.5, 1.0, 1.0], 0.0, 1.0, n)
        p = abi.Tf1dParams(lo, 1.0 / w, 0.0, 1.0 / w, 0.4, 0.6, 0.2, 10.0)
        return abi.TF1D(ctx, alpha, rgb, p, galpha=ga)
    return abi.TF1D(ctx, alpha, rgb, abi.Tf1dParams(lo, 1.0 / w, 0.0, float("inf"), 1.0, 0.0, 0.0, 1.0))


def _tf2d_tables(case, seed):
    """Opacity bumps over (intensity, gradient), the rest exactly empty."""
    r = _np_rng(case, seed, 6)
    n = case["n"]
    i, g = np.meshgrid(np.arange(n) / (n - 1.0), np.arange(n) / (n - 1.0))
    alpha, col, ws = np.zeros((n, n)), np.zeros((n, n, 3)), np.zeros((n, n))
    for ci, cg, a in ((0.3, 0.3, 0.05), (0.42, 0.6, 0.1), (0.55, 0.2, 0.2), (0.7, 0.75, 0.35), (0.85, 0.45, 0.6)):
        w = np.exp(-0.5 * (((i - ci - r.uniform(-0.02, 0.02)) / r.uniform(0.03, 0.05)) ** 2 +
                           ((g - cg - r.uniform(-0.05, 0.05)) / r.uniform(0.1, 0.2)) ** 2))
        alpha += a * r.uniform(0.9, 1.1) * w
        col += w[..., None] * r.uniform(0, 1, 3)
        ws += w
    alpha = np.clip(alpha, 0.0, 1.0)
    alpha[alpha < 0.004] = 0.0
    col /= np.maximum(ws, 1e-12)[..., None]
    full = np.ones((n, n))
    t = {"alpha": alpha, "red": col[..., 0], "green": col[..., 1], "blue": col[..., 2], "ambient": 0.4 * full,
         "diffuse": 0.6 * full, "specular": 0.2 * full, "specular_power": 12.0 * full}
    return {k: np.ascontiguousarray(v, np.float32) for k, v in t.items()}


def _tf2d_params(imin, imax, gmax):
    off = 0.8 * gmax
    top = math.log2(gmax * gmax + off) - math.log2(off) + 1.0
    return abi.Tf2dParams(imin, 1.0 / (imax - imin), -math.log2(off), 1.0 / top, off)


def _keyhole(view, case):
    """A window box in voxel space around the middle of the volume."""
    f = []
    for a, n in enumerate((case["nx"], case["ny"], case["nz"])):
        for sign, at in ((1.0, 0.25 * n), (-1.0, 0.75 * n)):
            p = [0.0, 0.0, 0.0, -sign * at]
            p[a] = sign
            f += p
    view.n_keyhole_planes = 6
    view.keyhole_planes[:] = f


@functools.lru_cache(maxsize=None)
def _context():
    """A program's one context; it outlives the handles made on it."""
    return abi.Context(0)


def prepare(case, seed):
    kind, sp = case["kind"], _spacing(case)
    dims = (case["nx"], case["ny"], case["nz"])
    ctx = _context()
    s = {"kind": kind, "case": case, "ctx": ctx}

    def volume(t, dtype):
        v = abi.Volume(ctx, dims, sp, dtype)
        v.set_frame(0, t)
        return v

    if kind in ("register", "poses", "reconstruct"):
        cams, sizes, poses = _poses(case, seed)
        march = abi.MarchParams(float(case["step"]), 0.0, 1, 0, 1)
        ct = _ct(case, seed)
        if kind == "reconstruct":
            s["renderer"] = DrrRenderer(_mu(ct), sp, [_abi_cam(c) for c in cams], sizes, _center(case), march,
                                        _drr_params(case), ctx=ctx)
            s["poses"] = torch.tensor(poses, dtype=torch.float64)
            s["volume"] = _iterate(ct, seed)
            s["target"] = torch.rand(s["renderer"].plan.total, device="cuda", generator=_gen(seed + 1))
        else:
            s["vol"] = volume(_mu(ct), np.float32) if kind == "register" else volume(ct, np.int16)
            vd = [abi.posed_view(_abi_cam(c), p, _center(case), w, h, spacing=sp, with_derivatives=True)
                  for c, p, (w, h) in zip(cams, poses, sizes)]
            plan = abi.DrrPlan(ctx, s["vol"], [v for v, _ in vd], march, _drr_params(case),
                               dview=np.stack([d for _, d in vd]))
            s["plan"] = plan
            s["out"] = torch.empty(plan.total, dtype=torch.float32, device="cuda")
            s["target"] = torch.rand(plan.total, device="cuda", generator=_gen(seed + 1))
            s["loss"] = torch.empty(plan.n_views, dtype=torch.float32, device="cuda")
            s["grad"] = torch.empty(plan.n_views * 6, dtype=torch.float32, device="cuda")
            if case.get("captured"):
                plan.capture(s["out"], s["target"], s["loss"], s["grad"])
        return s

    W, H = case["w"], case["h"]
    s["rgba"] = torch.empty((H, W, 4), dtype=torch.uint8, device="cuda")
    if kind == "drr":
        angle = _np_rng(case, seed, 7).uniform(0, 2 * math.pi)
        s["vol"] = volume(_ct(case, seed), np.int16)
        s["view"] = abi.compute_view(_abi_cam(_drr_cam(case, angle)), W, H, spacing=sp)
        s["march"], s["drr"] = _march(case, 0.0), _drr_params(case)
        if case["output"] != "rgba":
            s["out"] = torch.empty((H, W), dtype=torch.float32, device="cuda")
        return s

    s["view"] = abi.compute_view(_abi_cam(_scene_cam(case, seed)), W, H, spacing=sp)
    if kind == "tf1d":
        dt = case["dtype"]
        if dt == "u8":
            frame, lo, hi = _blobs(case, seed, 255.0, 10.0, False).round_().to(torch.uint8), 0.0, 255.0
        elif dt == "u16":
            frame, lo, hi = _blobs(case, seed, 4095.0, 0.0, True).round_().to(torch.uint16), 0.0, 4095.0
        elif dt == "f32":
            frame, lo, hi = _mu(_ct(case, seed)), 0.0, 0.05
        else:
            frame, lo, hi = _ct(case, seed), -1024.0, 1500.0
        s["vol"] = volume(frame, dt)
        s["tf"] = _tf1d(case, seed, ctx, lo, hi)
        s["march"] = _march(case, 0.01 if not case["shaded"] else 1.0 / 64.0)
        if case["live"]:
            s["frame"] = frame
    elif kind == "tf2d":
        gmax = 512.0
        s["vol"] = volume(_blobs(case, seed, 4095.0, 0.0, True).round_().to(torch.uint16), np.uint16)
        s["tf"] = abi.TF2D(ctx, _tf2d_tables(case, seed), _tf2d_params(0.0, 4095.0, gmax))
        if case["gradmag"]:
            s["vol"].compute_gradmag(0, gmax)
        s["march"] = _march(case, 0.01 if case["gradmag"] else 1.0 / 32.0)
        if case["post"]:
            s["depth"] = [torch.empty((H, W), dtype=torch.float32, device="cuda") for _ in range(3)]
            s["aux"] = abi.AuxOut(*[b.data_ptr() for b in s["depth"]])
            s["shade"] = abi.ShadeParams(0.7, 0.002, 1.0 / 0.003, 0.25, 0.45, 1.0 / 0.15)
    elif kind == "inex":
        s["vol"] = volume(_ct(case, seed), np.int16)
        tables = _tf2d_tables(case, seed)
        n = case["n"]
        cut, mark = int(0.3 * n), int(0.2 * n)  # above: excludes outside the keyhole; between: marks; below: empty
        tables["alpha"][:, :cut] = 0.0
        inex = np.zeros((n, n), np.float32)
        inex[:, cut:] = 1.0
        inex[:, mark:cut] = 0.3
        s["tf"] = abi.TF2D(ctx, tables, _tf2d_params(-1024.0, 1500.0, 512.0))
        s["tf"].set_inex(inex)
        if case["keyhole"]:
            _keyhole(s["view"], case)
        s["march"] = _march(case, 1.0 / 32.0)
    else:  # dual: two energies of one patient
        ct = _ct(case, seed)
        s["vol"] = volume(ct, np.int16)
        s["vol2"] = volume((ct.float() * 0.8 - 100.0).round_().to(torch.int16), np.int16)
        s["tf"] = abi.TF2D(ctx, _tf2d_tables(case, seed), _tf2d_params(-1024.0, 1500.0, 512.0))
        s["dual"] = abi.DualParams(-1024.0, 1.0 / 2524.0, -1024.0, 1.0 / 2524.0)
        s["march"] = _march(case, 1.0 / 32.0)
    return s


def _iterate(ct, seed):
    """An attenuation volume as an optimiser would have it: noise on top."""
    mu = _mu(ct)
    mu.mul_(torch.rand(mu.shape, device="cuda", generator=_gen(seed + 2)).mul_(0.2).add_(0.9))
    return mu


def run(state):
    s, kind, ctx = state, state["kind"], state["ctx"]
    if kind == "drr":
        out = s.get("out", s["rgba"])
        abi.render_drr(ctx, s["vol"], s["view"], s["march"], s["drr"], out)
        return out
    if kind == "tf1d":
        if "frame" in s:
            s["vol"].set_frame(0, s["frame"])
        abi.render_1d(ctx, s["vol"], s["tf"], s["view"], s["march"], s["rgba"])
        return s["rgba"]
    if kind == "tf2d":
        abi.render_2d(ctx, s["vol"], s["tf"], s["view"], s["march"], s["rgba"], s["case"]["gradmag"], s.get("aux"))
        if "aux" not in s:
            return s["rgba"]
        d = s["depth"]
        h, w = d[0].shape
        abi.check(abi.lib().rvk_post_shade(ctx.handle, w, h, s["shade"], d[0].data_ptr(), d[1].data_ptr(),
                                           d[2].data_ptr(), s["rgba"].data_ptr()))
        return [s["rgba"], *d]
    if kind == "inex":
        abi.render_2d_inex(ctx, s["vol"], s["tf"], s["view"], s["march"], s["rgba"], s["case"]["keyhole"])
        return s["rgba"]
    if kind == "dual":
        abi.render_dual(ctx, s["vol"], s["vol2"], s["tf"], s["dual"], s["view"], s["march"], s["rgba"])
        return s["rgba"]
    if kind == "register":
        s["plan"].register(s["out"], s["target"], s["loss"], s["grad"])
        return [s["out"], s["loss"], s["grad"]]
    if kind == "poses":
        s["plan"].render(s["out"])
        dldi = s["out"] - s["target"]
        s["plan"].backward(s["out"], dldi, grad_pose=s["grad"])
        return [s["out"], s["grad"]]
    poses = s["poses"].detach().requires_grad_(True)
    volume = s["volume"].detach().requires_grad_(True)
    images = drr_render(s["renderer"], poses, volume)
    images.backward(images.detach() - s["target"])
    return [images.detach(), volume.grad, poses.grad]


# ---------------------------------------------------------------------------
# what one pass cannot do without
def _chord_samples(case, cam, w, h, pose=None):
    """Samples of the plain march, from the chords of a 48 x 48 grid of
    rays through the crop box [1, n - 2]."""
    m = _matrix64(case, cam, w, h, pose).cpu().numpy()
    g = (np.arange(48) + 0.5) / 48.0
    vx, vy = (a.ravel() for a in np.meshgrid(g, g))
    pt = []
    for z in (0.0, 1.0):
        q = np.stack([vx, vy, np.full_like(vx, z), np.ones_like(vx)], 0)
        r = m @ q
        pt.append(r[:3] / r[3])
    s, d = pt[0], pt[1] - pt[0]
    n = np.array([[case["nx"]], [case["ny"]], [case["nz"]]], float)
    with np.errstate(divide="ignore", invalid="ignore"):
        ta, tb = (1.0 - s) / d, (n - 2.0 - s) / d
    t0 = np.maximum(np.nanmax(np.minimum(ta, tb), 0), 0.0)
    t1 = np.minimum(np.nanmin(np.maximum(ta, tb), 0), 1.0)
    sp = np.array(_spacing(case))[:, None]
    length = np.maximum(t1 - t0, 0.0) * np.sqrt(((d * sp) ** 2).sum(0))
    return float(length.mean()) / (min(_spacing(case)) * case["step"]) * w * h


def work(case):
    """Bytes: each voxel read once at its own type, each output written once
    (inputs of the gradients read once).  Flops: 14 for the trilinear value
    and 7 for position and accumulation per sample of the march; 16 more per
    sample for a pose gradient and 24 for a volume gradient."""
    kind = case["kind"]
    vox = case["nx"] * case["ny"] * case["nz"]
    if kind in ("register", "poses", "reconstruct"):
        cams, sizes, poses = _poses(case, 0)
        n = sum(_chord_samples(case, c, w, h, p) for c, (w, h), p in zip(cams, sizes, poses))
        pix = sum(w * h for w, h in sizes)
        if kind == "register":
            return {"bytes": 4.0 * vox + 8.0 * pix, "flops": 37.0 * n}
        if kind == "poses":
            return {"bytes": 2.0 * vox + 8.0 * pix, "flops": 37.0 * n}
        return {"bytes": 8.0 * vox + 8.0 * pix, "flops": 61.0 * n}
    pix = case["w"] * case["h"]
    if kind == "drr":
        b, cam = 2, _drr_cam(case, 0.3)
    else:
        b = {"u8": 1, "f32": 4}.get(case.get("dtype"), 2)
        cam = _scene_cam(case, 0)
    n = _chord_samples(case, cam, case["w"], case["h"])
    if kind == "tf2d" and case["gradmag"]:
        b += 1
    if kind == "dual":
        b += 2
    out = 16.0 if case.get("post") else 4.0
    return {"bytes": float(b * vox) + out * pix, "flops": 21.0 * n}


# ---------------------------------------------------------------------------
# the float results in 64 bits
_OFFSETS = np.array([
    70554, 53342, 57951, 28956, 30194, 77474, 1401, 76072, 81449, 70903, 4535, 41403, 86261, 79048, 37353, 96195,
    87144, 5623, 94955, 36401, 52486, 76711, 5350, 59245, 46870, 29816, 62269, 64782, 26379, 27934, 82980, 82460,
    58916, 98609, 91096, 22686, 69511, 98000, 24393, 53387, 10636, 99941, 67617, 1570, 57518, 10005, 10302, 79888,
    28448, 4564, 29577, 38201, 30097, 94857, 97982, 40137, 27827, 16044, 16282, 64658, 41007, 41276, 71273, 32620,
    63317, 20756, 18601, 58335, 8071, 45797, 90572, 26136, 78521, 37890, 28966, 91937, 63174, 62764, 42845, 9797,
    56104, 69448, 91371, 83481, 2262, 54336, 91616, 43026, 67794, 50245, 51373, 46298, 35347, 40483, 26973, 5559,
    24384, 97907, 6091, 39029, 36499, 48989, 15566, 47445, 25726, 62875, 54207, 15630, 93854, 65449, 50608, 39047,
    10737, 78399, 45964, 75368, 59609, 83273, 1875, 21036, 7395, 10545, 33169, 12824, 24, 53679, 65705, 54401,
    82741, 8189, 19192, 67891, 45420, 35702, 14998, 70439, 92878, 53021, 8964, 75772, 40184, 46187, 49216, 20762,
    32973, 9542, 58979, 16987, 92761, 9792, 44386, 27294, 87254, 75068, 27294, 67364, 25662, 8989, 3095, 32271,
    79012, 29725, 23528, 48047, 25460, 34060, 4493, 48242, 20601, 86453, 58862, 75490, 92788, 33101, 54294, 8069,
    63437, 41003, 96042, 11462, 92344, 62020, 34772, 14924, 47997, 21940, 99373, 13042, 2888, 34539, 54766, 92295,
    53824, 40642, 84724, 82622, 67242, 72189, 99677, 33980, 49521, 41296, 69528, 17908, 42291, 54317, 81466, 54091,
    42753, 50906, 22778, 61918, 48983, 68081, 88660, 37051, 30249, 29286, 15031, 52982, 22326, 58452, 36345, 87597,
    47801, 19063, 68406, 74741, 61393, 78213, 16174, 80777, 20261, 95676, 6585, 6152, 79319, 37960, 46358, 11954,
    11547, 17377, 4811, 71481, 53302, 56100, 21673, 46800, 74635, 75231, 39893, 90309, 74600, 8855, 63457, 71302])


def _matrix64(case, cam, w, h, pose=None):
    """Screen -> voxel matrix of pixel coordinates vx = 1 - x/w, vy = y/h and
    depth 0..1, differentiable in the pose."""
    f64 = dict(dtype=torch.float64)
    n = cam["position"] - cam["focal"]
    n = n / np.linalg.norm(n)
    s = np.cross(cam["up"], n)
    s = s / np.linalg.norm(s)
    v = np.eye(4)
    v[0, :3], v[1, :3], v[2, :3] = s, np.cross(n, s), n
    v[:3, 3] = -v[:3, :3] @ cam["position"]
    t = math.tan(math.radians(cam["angle"]) / 2.0)
    near, far = cam["near"], cam["far"]
    p = np.zeros((4, 4))
    p[0, 0], p[1, 1] = 1.0 / (t * w / h), 1.0 / t
    p[2, 2], p[2, 3], p[3, 2] = -(near + far) / (far - near), -2.0 * near * far / (far - near), -1.0
    p[2] = 0.5 * p[2] + 0.5 * p[3]
    pv = torch.tensor(p @ v, **f64)
    vox = torch.diag(torch.tensor([*_spacing(case), 1.0], **f64))
    if pose is not None:
        pose = torch.as_tensor(pose, **f64)
        c = torch.tensor(_center(case), **f64)
        i3, rot = torch.eye(3, **f64), torch.eye(3, **f64)
        for a in range(3):  # Rz Ry Rx
            k = torch.zeros(3, 3, **f64)
            i, j = (a + 1) % 3, (a + 2) % 3
            k[i, j], k[j, i] = -1.0, 1.0
            rot = (i3 + torch.sin(pose[a]) * k + (1.0 - torch.cos(pose[a])) * (k @ k)) @ rot
        top = torch.cat([rot, (c + pose[3:] - rot @ c)[:, None]], 1)
        vox = torch.cat([top, torch.tensor([[0.0, 0.0, 0.0, 1.0]], **f64)], 0) @ vox
    m = torch.linalg.inv(pv @ vox)
    return torch.stack([-2.0 * m[:, 0], 2.0 * m[:, 1], m[:, 2], m[:, 3] + m[:, 0] - m[:, 1]], 1)


def _rays64(case, m, w, h):
    """First sample, step vector and step count (real) of every ray."""
    dev = dict(dtype=torch.float64, device="cuda")
    y, x = torch.meshgrid(torch.arange(h, device="cuda"), torch.arange(w, device="cuda"), indexing="ij")
    j = torch.tensor(_OFFSETS * 1e-5, **dev)[((x % 16) + 16 * (y % 16)).reshape(-1)]
    vx, vy = 1.0 - x.reshape(-1).double() / w, y.reshape(-1).double() / h

    def at(z):
        q = [vx * m[r, 0] + vy * m[r, 1] + z * m[r, 2] + m[r, 3] for r in range(4)]
        return [q[r] / q[3] for r in range(3)]

    s, e = at(0.0), at(1.0)
    n = (case["nx"], case["ny"], case["nz"])
    zero = torch.zeros_like(vx)
    d = [b - a for a, b in zip(s, e)]
    for a in range(3):  # crop to [1, n - 2] axis by axis; d stays that of the uncropped ray
        lo, hi = 1.0, n[a] - 2.0
        up = d[a] > 0
        ds = torch.where(up, torch.where(s[a] < lo, lo - s[a], zero), torch.where(s[a] > hi, hi - s[a], zero)) / d[a]
        de = torch.where(up, torch.where(e[a] > hi, hi - e[a], zero), torch.where(e[a] < lo, lo - e[a], zero)) / d[a]
        s = [p + q * ds for p, q in zip(s, d)]
        e = [p + q * de for p, q in zip(e, d)]
    out = torch.zeros_like(vx, dtype=torch.bool)
    for a in range(3):
        for p in (s[a], e[a]):
            out = out | (p > n[a] - 1.0) | (p < 0.0)
    s = [torch.where(out, q, p) for p, q in zip(s, e)]
    sp = _spacing(case)
    d = [b - a for a, b in zip(s, e)]
    q = sum((k * c) ** 2 for k, c in zip(d, sp))
    hit = q > 0
    ns = torch.sqrt(torch.where(hit, q, torch.ones_like(q))) / (min(sp) * case["step"])
    inc = [torch.where(hit, k / ns, zero) for k in d]
    start = [torch.where(hit, a, zero) for a in s]
    return start, inc, torch.where(hit, ns, zero), j


def _depths64(case, m, w, h):
    """Where each ray enters and leaves, in voxels from the near plane; a ray
    past the volume enters where it leaves."""
    start, _, ns, _ = _rays64(case, m, w, h)
    y, x = torch.meshgrid(torch.arange(h, device="cuda"), torch.arange(w, device="cuda"), indexing="ij")
    vx, vy = 1.0 - x.reshape(-1).double() / w, y.reshape(-1).double() / h
    q = [[vx * m[r, 0] + vy * m[r, 1] + z * m[r, 2] + m[r, 3] for r in range(4)] for z in (0.0, 1.0)]
    near, far = [[a[r] / a[3] for r in range(3)] for a in q]
    last = torch.sqrt(sum((b - a) ** 2 for a, b in zip(near, far)))
    first = torch.where(ns > 0, torch.sqrt(sum((b - a) ** 2 for a, b in zip(near, start))), last)
    return first.reshape(h, w), last.reshape(h, w)


def _cells64(vol, p, case):
    """Clamped indices of the 8 voxels around p and the weights' fractions."""
    n = (case["nx"], case["ny"], case["nz"])
    i, f = [], []
    for a in range(3):
        c = p[a] + 0.5
        k = torch.floor(c)
        f.append(c - k)
        k = k.long()
        i.append(((k - 1).clamp(0, n[a] - 1), k.clamp(0, n[a] - 1)))
    rows = [[(i[2][z] * n[1] + i[1][y]) * n[0] for y in range(2)] for z in range(2)]
    return [rows[z][y] + i[0][x] for z in range(2) for y in range(2) for x in range(2)], f


def _march64(case, vol, rays, cs0, ci0, skip, grads=False, scatter=None):
    """Line integral L of every ray; with grads the sums of the sample
    gradients A and of (offset + index) times them B; with scatter =
    (target, coefficient) the adjoint of the samples added to target."""
    start, inc, ns, j = rays
    kst = torch.floor(ns - j).clamp(min=0)
    sp = _spacing(case)
    ds = torch.sqrt(sum((k * c) ** 2 for k, c in zip(inc, sp)))
    keep = torch.nonzero(kst > 0).reshape(-1)
    L = torch.zeros_like(ds)
    A = [torch.zeros_like(ds) for _ in range(3)] if grads else None
    B = [torch.zeros_like(ds) for _ in range(3)] if grads else None
    if keep.numel() == 0:
        return L, A, B
    p0 = [(s + j * k)[keep] for s, k in zip(start, inc)]
    inc, kst, dsk, jk = [k[keep] for k in inc], kst[keep], ds[keep], j[keep]
    coef = scatter[1][keep] if scatter else None
    acc = torch.zeros_like(dsk)
    a_, b_ = ([torch.zeros_like(dsk) for _ in range(3)] for _ in range(2))
    t, back, skipped = torch.zeros_like(dsk), torch.zeros_like(dsk, dtype=torch.bool), None
    skipped = torch.zeros_like(back)
    steps = 0
    while True:
        live = t < kst
        steps += 1
        if steps % 32 == 1 and not bool(live.any()):
            break
        idx, f = _cells64(vol, [a + t * k for a, k in zip(p0, inc)], case)
        v = [vol[k] for k in idx]
        x = [v[2 * k] + f[0] * (v[2 * k + 1] - v[2 * k]) for k in range(4)]
        yv = [x[0] + f[1] * (x[1] - x[0]), x[2] + f[1] * (x[3] - x[2])]
        mu = cs0 * (yv[0] + f[2] * (yv[1] - yv[0])) + ci0
        hit = live & (mu > 0)
        add = hit & ~skipped if skip else hit
        acc += torch.where(add, mu, torch.zeros_like(mu))
        if grads:
            dx = [v[2 * k + 1] - v[2 * k] for k in range(4)]
            dx0, dx1 = dx[0] + f[1] * (dx[1] - dx[0]), dx[2] + f[1] * (dx[3] - dx[2])
            g = [dx0 + f[2] * (dx1 - dx0), (x[1] - x[0]) + f[2] * ((x[3] - x[2]) - (x[1] - x[0])), yv[1] - yv[0]]
            for a in range(3):
                ga = torch.where(add, g[a], torch.zeros_like(mu))
                a_[a] += ga
                b_[a] += (jk + t) * ga
        if scatter:
            wz, wy, wx = ((1 - f[k], f[k]) for k in (2, 1, 0))
            c = torch.where(add, coef, torch.zeros_like(mu))
            for z in range(2):
                for y in range(2):
                    cy = c * wz[z] * wy[y]
                    for xx in range(2):
                        scatter[0].index_add_(0, idx[4 * z + 2 * y + xx], cy * wx[xx])
        if skip:
            # a contributing sample after a skipped one steps back; an empty one steps over its successor
            step = torch.where(hit, torch.where(skipped, -1.0, 1.0), torch.where(back, 1.0, 2.0))
            back, skipped = hit & skipped, ~hit & ~back
            t = t + step.double()
        else:
            t = t + 1.0
    L[keep] = acc * dsk
    if grads:
        for a in range(3):
            A[a][keep], B[a][keep] = a_[a] * dsk * cs0, b_[a] * dsk * cs0
    return L, A, B


def _pose_grad64(case, cam, w, h, pose, A, B, coef):
    """Sum over pixels of coef * dL/d pose."""
    def geometry(q):
        start, inc, _, _ = _rays64(case, _matrix64(case, cam, w, h, q).cuda(), w, h)
        return torch.stack(start + inc)

    q = torch.as_tensor(pose, dtype=torch.float64)
    ab = torch.stack(A + B)
    out = []
    for i in range(6):
        _, d = torch.func.jvp(geometry, (q,), (torch.eye(6, dtype=torch.float64)[i],))
        out.append((coef * torch.where(ab != 0, ab * d, torch.zeros_like(d)).sum(0)).sum())
    return torch.stack(out)


def exact(case, seed):
    kind = case["kind"]
    if kind == "drr" and case["output"] != "rgba":
        angle = _np_rng(case, seed, 7).uniform(0, 2 * math.pi)
        cam, w, h = _drr_cam(case, angle), case["w"], case["h"]
        vol = _ct(case, seed).reshape(-1).double()
        L, _, _ = _march64(case, vol, _rays64(case, _matrix64(case, cam, w, h).cuda(), w, h), 2e-5, 0.02,
                           case["skip"])
        return (torch.exp(-L) if case["output"] == "exp" else L).reshape(h, w)
    if kind == "tf2d" and case["post"]:
        return [None, None, *_depths64(case, _matrix64(case, _scene_cam(case, seed), case["w"], case["h"]).cuda(),
                                       case["w"], case["h"])]
    if kind not in ("register", "poses", "reconstruct") or work(case)["flops"] > 2.5e11:
        return None
    cams, sizes, poses = _poses(case, seed)
    ct = _ct(case, seed)
    total = sum(w * h for w, h in sizes)
    target = torch.rand(total, device="cuda", generator=_gen(seed + 1)).double()
    cs, ci = (2e-5, 0.02) if kind == "poses" else (1.0, 0.0)
    vol = (ct if kind == "poses" else _mu(ct) if kind == "register" else _iterate(ct, seed)).reshape(-1).double()
    images, losses, gposes, at = [], [], [], 0
    gvol = torch.zeros_like(vol) if kind == "reconstruct" else None
    for cam, (w, h), pose in zip(cams, sizes, poses):
        rays = _rays64(case, _matrix64(case, cam, w, h, pose).cuda(), w, h)
        L, A, B = _march64(case, vol, rays, cs, ci, False, grads=True)
        img, tgt = torch.exp(-L), target[at:at + w * h]
        at += w * h
        if kind == "register":
            a, b = img - img.mean(), tgt - tgt.mean()
            saa, sbb, sab = (a * a).sum(), (b * b).sum(), (a * b).sum()
            ncc = sab / torch.sqrt(saa * sbb)
            losses.append(1.0 - ncc)
            dldi = -(b / torch.sqrt(saa * sbb) - ncc * a / saa)
        else:
            dldi = img - tgt
        coef = -dldi * img
        gposes.append(_pose_grad64(case, cam, w, h, pose, A, B, coef))
        if kind == "reconstruct":
            ds = torch.sqrt(sum((k * c) ** 2 for k, c in zip(rays[1], _spacing(case))))
            _march64(case, vol, rays, cs, ci, False, scatter=(gvol, coef * ds * cs))
        images.append(img)
    images, gp = torch.cat(images), torch.stack(gposes)
    if kind == "register":
        return [images, torch.stack(losses), gp.reshape(-1)]
    if kind == "poses":
        return [images, gp.reshape(-1)]
    return [images, gvol.reshape(case["nz"], case["ny"], case["nx"]), gp.cpu()]
