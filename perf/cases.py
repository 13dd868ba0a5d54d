"""The measured workloads of blacktracer_amd: what a program that uses the
package has it do, through its public entry points.

    rays        Grid::integration_wrapper on host arrays (trace_rays)
    sky         the same on device arrays: an equal-angle camera sky
    grid        one adaptive grid, built and read back (Grid, cel/steps/levels)
    batch       the grids of several cameras, built in one call and read back
    frame       one frame of a resident grid, scene and view
    blend       a frame between the grids of two camera positions
    trails      a sequence of frames with star trails and a diffraction sprite
    make_image  the one-shot makeImage call on host arrays

A case is a dict of plain values; a seed moves the camera a little, and
draws the rays, stars, sky and frame offset.
"""
import ctypes
import math
import random

import numpy as np
import torch

import blacktracer_amd as bt
from blacktracer_amd import _lib, scene

PI = 3.141592653589793238
FLOPS_PER_ATTEMPT = 1115       # one Cash-Karp attempt as the reference writes it
ATTEMPTS = 36                  # mean attempts of a ray at the reference settings
ATTEMPTS_RADIUS_STOP = 62      # ... at relative tolerance 1e-8 with radius stops


def listed():
    pose = {"a": 0.999, "r": 5.0, "theta": PI / 2}
    return [
        # a probe of a few hundred directions, as an interactive tool or a
        # unit check sends: latency counts
        {"name": "rays 500", "kind": "rays", "n": 500, "mode": "fp64", **pose},
        # the radius-stop settings (relative tolerance 1e-8, r > 1000 M or
        # the horizon), an odd count, off the equator
        {"name": "rays 20011 radius stop", "kind": "rays", "n": 20011, "mode": "radius", "a": 0.9, "r": 20.0,
         "theta": 1.1},
        # the quarter-size uniform sky on the plain FP64 path
        {"name": "sky 1025 fp64", "kind": "sky", "rows": 1025, "mode": "fp64", **pose},
        # the full uniform sky of the precision workload, mixed precision
        {"name": "sky 2049 mixed", "kind": "sky", "rows": 2049, "mode": "mixed", **pose},
        # the grid that a new camera position needs before its first frame
        {"name": "grid 10", "kind": "grid", "level": 10, "start": 1, "full": True, "mode": "fp64", **pose},
        # the grids of an orbit prepared together
        {"name": "batch 12", "kind": "batch", "count": 12, "low": 6, "high": 9, "full": True, "mode": "fp64"},
        # a thumbnail, the standard frame and the largest one served
        {"name": "frame 320x180", "kind": "frame", "w": 320, "h": 180, "step": 1, "star": True, "map": True,
         "stars": 100000, "cols": 4096, "level": 9, **pose},
        {"name": "frame 1920x1080", "kind": "frame", "w": 1920, "h": 1080, "step": 1, "star": True, "map": True,
         "stars": 100000, "cols": 4096, "level": 10, **pose},
        {"name": "frame 3840x2160", "kind": "frame", "w": 3840, "h": 2160, "step": 1, "star": True, "map": True,
         "stars": 100000, "cols": 4096, "level": 10, "a": 0.5, "r": 12.0, "theta": 1.3},
        # the display loop between two cached grids
        {"name": "blend 1440x810", "kind": "blend", "w": 1440, "h": 810, "step": 1, "stars": 100000, "cols": 4096,
         "level": 9, **pose},
        # the display loop's effects over four consecutive frames
        {"name": "trails 1366x768", "kind": "trails", "w": 1366, "h": 768, "step": 1, "frames": 4, "sprite": True,
         "stars": 100000, "cols": 4096, "level": 9, **pose},
        # the drop-in of the reference's makeImage: everything from the host
        {"name": "make_image 1920x1080", "kind": "make_image", "w": 1920, "h": 1080, "step": 1, "stars": 100000,
         "cols": 4096, "level": 9, **pose},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    pose = {"a": round(rng.uniform(0.01, 0.999), 4), "r": round(math.exp(rng.uniform(math.log(3.0), math.log(50.0))), 3),
            "theta": round(rng.uniform(0.1, PI - 0.1), 4)}
    kind = rng.choice(["rays", "sky", "grid", "batch", "frame", "frame", "blend", "trails", "make_image"])
    mode = rng.choice(["fp64", "mixed"])
    if kind == "rays":
        n = _log_uniform(rng, 1, 200000)
        return {"kind": kind, "n": n, "mode": rng.choice(["fp64", "mixed", "radius"]), **pose}
    if kind == "sky":
        return {"kind": kind, "rows": _log_uniform(rng, 129, 1400), "mode": mode, **pose}
    if kind == "grid":
        start = rng.randint(1, 5)
        return {"kind": kind, "level": rng.randint(max(5, start), 10), "start": start, "full": rng.random() < 0.7,
                "mode": mode, **pose}
    if kind == "batch":
        low = rng.randint(4, 8)
        return {"kind": kind, "count": rng.randint(2, 12), "low": low, "high": rng.randint(low, 9),
                "full": rng.random() < 0.7, "mode": mode}
    w = _log_uniform(rng, 160, 2560 if kind != "frame" else 3840)
    h = max(90, min(2160, int(w * rng.choice([9 / 16, 9 / 16, 0.75, 0.6]))))
    # the default view looks from the equatorial plane at +-45 degrees
    case = {"kind": kind, "w": w, "h": h, "step": 1, "stars": _log_uniform(rng, 5000, 150000),
            "cols": rng.choice([1024, 2048, 4096]), "level": rng.randint(8, 10), **pose}
    if kind == "frame":
        star, sky = rng.choice([(True, True), (True, True), (True, False), (False, True)])
        case.update(star=star, map=sky, step=rng.choice([1, 1, 2]))
    elif kind == "trails":
        case.update(frames=rng.randint(2, 4), sprite=rng.random() < 0.5)
    return case


# ------------------------------------------------------------------ inputs


def _camera(a, r, theta, rng):
    """A camera near (r, theta) of the case, as the seed has it."""
    hole = bt.BlackHole(a)
    theta = min(max(theta + 0.01 * (rng.random() - 0.5), 0.05), PI - 0.05)
    return bt.Camera(theta, 0.0, r * (1 + 0.01 * (rng.random() - 0.5)), black_hole=hole), hole


def _params(mode):
    if mode == "radius":
        return bt.radius_stop_params()
    return bt.IntegParams(bt.BT_PREC_MIXED if mode == "mixed" else bt.BT_PREC_FP64)


def _sky_image(cols, seed):
    """(cols / 2, cols, 3) uint8 BGR: smooth noise on three scales over a band."""
    gen = torch.Generator().manual_seed(seed)
    rows = cols // 2
    img = torch.zeros(1, 3, rows, cols)
    for cells, weight in ((16, 0.5), (64, 0.3), (256, 0.2)):
        coarse = torch.rand(1, 3, cells // 2, cells, generator=gen)
        img += weight * torch.nn.functional.interpolate(coarse, size=(rows, cols), mode="bilinear", align_corners=False)
    band = torch.exp(-((torch.arange(rows) + 0.5 - rows / 2) / (0.12 * rows)) ** 2).view(1, 1, rows, 1)
    img = (20 + 60 * img + 150 * band * img).clamp(0, 255)
    return img[0].permute(1, 2, 0).to(torch.uint8).contiguous().numpy()


class _Frame:
    """A device frame buffer held by torch; ptr is what the package takes."""

    def __init__(self, w, h):
        self.pixels = torch.zeros((h, w, 4), dtype=torch.uint8, device="cuda")
        self.ptr = ctypes.c_void_p(self.pixels.data_ptr())


def prepare(case, seed):
    rng = random.Random(seed)
    kind = case["kind"]
    st = {"kind": kind, "case": case}
    if kind == "batch":
        cams = []
        for _ in range(case["count"]):
            cams.append(_camera(rng.uniform(0.01, 0.999), rng.uniform(3, 50), rng.uniform(0.1, PI - 0.1), rng))
        levels = [case["low"] + k % (case["high"] - case["low"] + 1) for k in range(case["count"])]
        st.update(cams=[c for c, _ in cams], holes=[b for _, b in cams], levels=levels,
                  starts=[1] * case["count"], params=_params(case["mode"]))
        return st
    cam, hole = _camera(case["a"], case["r"], case["theta"], rng)
    st.update(cam=cam, hole=hole)
    if kind == "rays":
        g = np.random.default_rng(seed)
        st.update(theta=np.arccos(1 - 2 * g.random(case["n"])), phi=2 * PI * g.random(case["n"]),
                  params=_params(case["mode"]))
        return st
    if kind == "sky":
        rows = case["rows"]
        cols = 2 * (rows - 1)
        ti = (torch.arange(rows, dtype=torch.float64, device="cuda") + 0.9 * rng.random()) / rows * PI
        pj = (torch.arange(cols, dtype=torch.float64, device="cuda") + rng.random()) / cols * (2 * PI)
        st.update(theta0=ti.repeat_interleave(cols), phi0=pj.repeat(rows), params=_params(case["mode"]),
                  ctx=bt.default_context(), pose=cam.pose())
        st.update(theta=torch.empty_like(st["theta0"]), phi=torch.empty_like(st["phi0"]),
                  step=torch.empty(rows * cols, dtype=torch.int32, device="cuda"))
        return st
    if kind == "grid":
        st.update(params=_params(case["mode"]))
        return st
    # the frames: grid(s), stars, sky, view
    w, h = case["w"], case["h"]
    stars = scene.synthetic_stars(case["stars"], seed=seed)
    sky = _sky_image(case["cols"], seed)
    grid = bt.Grid(case["level"], 1, True, cam, hole)
    st.update(offset=0.5 * rng.random(), out=_Frame(w, h))
    if kind == "make_image":
        tree, pos, mag = bt.star_tree(stars, 8)
        ht, ot, tag, hw, ow = grid.psh()
        st.update(args=(pos, tree, cam.getParamArray(), mag, 8, w, h, case["step"], sky,
                        bt.viewer_matrix(PI / 2, 0.0, PI / 16, w, h), grid.M, grid.N, case["level"], ot, ht, tag, hw,
                        ow))
        return st
    st.update(grid=grid, scene=bt.Scene(stars, sky, tree_level=8), view=bt.View(w, h))
    if kind == "blend":
        cam2 = bt.Camera(cam.theta, 0.0, cam.r * 1.04, black_hole=hole)
        st.update(grid2=bt.Grid(case["level"], 1, True, cam2, hole), alpha=0.2 + 0.6 * rng.random())
    if kind == "trails":
        sprite = None
        if case["sprite"]:
            fs = w // 16
            y, x = np.mgrid[0:fs, 0:fs] - (fs - 1) / 2
            glow = 255 * np.exp(-(x * x + y * y) / (0.06 * fs * fs)) * (0.3 + 0.7 * np.exp(-np.minimum(x * x, y * y) / 4))
            sprite = np.repeat(glow[..., None], 3, axis=2).astype(np.uint8)
        st.update(trails=bt.Trails(st["scene"], w, h, sprite), outs=[_Frame(w, h) for _ in range(case["frames"])])
    return st


# -------------------------------------------------------------------- runs


def run(st):
    kind, case = st["kind"], st["case"]
    if kind == "rays":
        return bt.trace_rays(st["cam"], st["theta"], st["phi"], params=st["params"])
    if kind == "sky":
        # the trace is in place: the directions are put back, and handed over
        # from torch's stream to the context's and back
        st["theta"].copy_(st["theta0"])
        st["phi"].copy_(st["phi0"])
        torch.cuda.current_stream().synchronize()
        _lib.check(_lib.load().bt_trace_rays_device(
            st["ctx"].handle, ctypes.byref(st["pose"]), ctypes.byref(st["params"]), st["theta"].numel(),
            st["theta"].data_ptr(), st["phi"].data_ptr(), st["step"].data_ptr(), None))
        st["ctx"].sync()
        return st["theta"], st["phi"], st["step"]
    if kind == "grid":
        g = bt.Grid(case["level"], case["start"], case["full"], st["cam"], st["hole"], params=st["params"])
        out = g.cel, g.steps, g.levels, g.rays_traced
        g.close()
        return out
    if kind == "batch":
        grids, _ = bt.Grid.build_batch(st["cams"], st["holes"], st["levels"], st["starts"], angle=case["full"],
                                       params=st["params"])
        out = [(g.cel, g.steps, g.levels, g.rays_traced) for g in grids]
        for g in grids:
            g.close()
        return out
    if kind == "make_image":
        return bt.make_image(*st["args"], flags=bt.RenderFlags(offset=st["offset"]))
    if kind == "frame":
        flags = bt.RenderFlags(star=case["star"], map=case["map"], offset=st["offset"])
        bt.render_frame_device(st["grid"], st["scene"], st["view"], st["out"], flags=flags, step=case["step"])
        return st["out"].pixels
    if kind == "blend":
        bt.render_frame_blend(st["grid"], st["grid2"], st["alpha"], st["scene"], st["view"],
                              flags=bt.RenderFlags(offset=st["offset"]), step=case["step"], out_buffer=st["out"])
        return st["out"].pixels
    # a sequence from its first frame, the sky turning by about two pixels a frame
    st["trails"].reset()
    for k, out in enumerate(st["outs"]):
        flags = bt.RenderFlags(offset=st["offset"] + k * 3.0 / case["w"])
        st["trails"].render(st["grid"], st["scene"], st["view"], flags=flags, step=case["step"], out_buffer=out)
    return [out.pixels for out in st["outs"]]


# -------------------------------------------------------------------- work


def _grid_points(level, full):
    """Grid points of a level, and rays an adaptive build of it traces (each
    level of refinement follows curves: about twice as many per level)."""
    n = 2 ** level // (1 if full else 2) + 1
    m = 2 * 2 ** level
    return n * m, min(n * m, 93 * 2 ** level)


def work(case):
    kind = case["kind"]
    per_ray = FLOPS_PER_ATTEMPT * (ATTEMPTS_RADIUS_STOP if case.get("mode") == "radius" else ATTEMPTS)
    if kind in ("rays", "sky"):
        n = case["n"] if kind == "rays" else case["rows"] * 2 * (case["rows"] - 1)
        return {"bytes": 36 * n, "flops": per_ray * n}
    if kind in ("grid", "batch"):
        levels = [case["level"]] if kind == "grid" else [
            case["low"] + k % (case["high"] - case["low"] + 1) for k in range(case["count"])]
        pts = [_grid_points(lv, case["full"]) for lv in levels]
        return {"bytes": 21 * sum(p for p, _ in pts), "flops": per_ray * sum(r for _, r in pts)}
    # frames: the grid, the stars, the view, two table reads per sky column
    # of every pixel's footprint (about seven columns of the sky per frame
    # row and sky column), the frame
    w, h = case["w"], case["h"]
    px = w * h
    pts = _grid_points(case["level"], True)[0]
    frame = 8 * pts + 16 * case["stars"] + 12 * px + 4 * px
    if case.get("map", True):
        frame += 32 * max(px, int(6.6 * h * case["cols"]))
    flops = 700 * px
    if kind == "blend":
        frame += 8 * pts
    if kind == "trails":
        frame, flops = case["frames"] * frame, case["frames"] * flops
    if kind == "make_image":
        table = case["cols"] * case["cols"] // 2
        frame += 19 * table + 24 * _grid_points(case["level"], True)[1]
        flops += 150 * table
    return {"bytes": frame, "flops": flops}


# ------------------------------------------------------------------- exact
# The ray batch in plain torch, FP64: initial conditions (Grid.h:524-547),
# the a-priori capture test (Metric.h:110-174) and the Cash-Karp integration
# with its step control (Metric.h:198-324).


def exact(case, seed):
    if case["kind"] not in ("rays", "sky"):
        return None       # adaptive grids end in ordered repairs, frames in bytes
    st = prepare(case, seed)
    p = st["params"]
    if case["kind"] == "rays":
        th, ph = (torch.from_numpy(st[k]).cuda() for k in ("theta", "phi"))
    else:
        th, ph = st["theta0"], st["phi0"]
    out = _trace(st["cam"].a, st["cam"].r, st["cam"].theta, th, ph, p)
    return out[0], out[1], None


def _pose(a, r, th):
    f32 = np.float32
    asq = a * a
    delta = r * r - 2 * r + asq
    sigma = math.sqrt((r * r + asq) ** 2 - asq * delta * math.sin(th) ** 2)
    ro = math.sqrt(r * r + asq * math.cos(th) ** 2)
    w, wbar, alpha = 2 * a * r / sigma ** 2, sigma * math.sin(th) / ro, ro * math.sqrt(delta) / sigma
    speed = wbar / alpha * (1 / (a + r ** 1.5) - w)
    r1, r2 = (2 * (1 + math.cos(2 * math.acos(s * a) / 3)) for s in (-1, 1))

    def b0(x):
        return -(x ** 3 - 3 * x * x + asq * x + asq) / (a * (x - 1))
    return dict(ro=ro, w=w, wbar=wbar, alpha=alpha, speed=speed, b1=b0(r2), b2=b0(r1),
                neg_s=-float(np.sqrt(f32(1 - speed * speed))), sqrt_d=float(np.sqrt(f32(delta))))


def _derivs(a, v, b, q):
    r, th, pr, pt = v[0], v[1], v[3], v[4]
    s, c = torch.sin(th), torch.cos(th)
    c2, s2 = c * c, s * s
    delta = r * r - 2 * r + a * a
    rho2 = r * r + a * a * c2
    P = r * r + a * a - a * b
    part = q + (a - b) ** 2
    R = P * P - delta * part
    bt_ = q - c2 * (b * b / s2 - a * a)
    bdr = bt_ * delta + R
    r4 = (2 * rho2) ** 2
    rd = rho2 * rho2 * delta
    two = 2 * r - 2
    acs = a * a * c * s
    return [delta / rho2 * pr,
            pt / rho2,
            (2 * a * P - (2 * a - 2 * b) * delta + 2 * b * c2 * delta / s2) / (2 * rho2 * delta),
            (two * bt_ - two * part + 4 * r * P) / (2 * rho2 * delta) - pr * pr * two / (2 * rho2)
            + 4 * pt * pt * r / r4 - (4 * r - 4) * bdr / (rho2 * (2 * delta) ** 2) + 4 * pr * pr * r * delta / r4
            - r * bdr / rd,
            (2 * c * s * (b * b / s2 - a * a) + 2 * b * b * c ** 3 / s ** 3) * delta / (2 * rho2 * delta)
            - 4 * acs * pt * pt / r4 - 4 * acs * pr * pr * delta / r4 + acs * bdr / rd]


_A = ((0.2,), (3 / 40, 9 / 40), (0.3, -0.9, 1.2), (-11 / 54, 2.5, -70 / 27, 35 / 27),
      (1631 / 55296, 175 / 512, 575 / 13824, 44275 / 110592, 253 / 4096))
_C = (37 / 378, 0.0, 250 / 621, 125 / 594, 0.0, 512 / 1771)
_D = (37 / 378 - 2825 / 27648, 0.0, 250 / 621 - 18575 / 48384, 125 / 594 - 13525 / 55296, -277 / 14336,
      512 / 1771 - 0.25)


def _combine(coef, ks, i):
    acc = None
    for x, k in zip(coef, ks):
        if x:
            acc = x * k[i] if acc is None else acc + x * k[i]
    return acc


def _escapes(pose, a, r, pr, b, q):
    """checkCelest: whether the ray came from the sky."""
    asq = a * a
    r0 = torch.full_like(b, 2.0)
    last = torch.full_like(b, 100.0)
    for _ in range(5000):
        go = (b - last).abs() > 1e-7
        if not bool(go.any()):
            break
        b0 = -(r0 ** 3 - 3 * r0 * r0 + asq * r0 + asq) / (a * (r0 - 1))
        d0 = (asq + a - 2 * r0 * (r0 * r0 - 3 * r0 + 3)) / (a * (r0 - 1) ** 2)
        new = r0 - (b0 - b) / d0
        last = torch.where(go, b0, last)
        r0 = torch.where(go, torch.where(new < 1, torch.full_like(new, 1.0001), new), r0)
    q0 = -r0 ** 3 * (r0 ** 3 - 6 * r0 * r0 + 9 * r0 - 4 * asq) / (asq * (r0 - 1) ** 2)
    outside = (pose["b1"] >= b) | (pose["b2"] <= b) | (q >= q0)

    def big_r(x):
        return (x * x + asq - a * b) ** 2 - (x * x - 2 * x + asq) * ((b - a) ** 2 + q)
    golden = (math.sqrt(5.0) + 1) / 2
    lo, hi = torch.full_like(b, r), torch.full_like(b, 4 * r)
    c, d = hi - (hi - lo) / golden, lo + (hi - lo) / golden
    for _ in range(200):
        go = (c - d).abs() > 1e-5
        if not bool(go.any()):
            break
        left = big_r(c) < big_r(d)
        hi, lo = torch.where(go & left, d, hi), torch.where(go & ~left, c, lo)
        c, d = hi - (hi - lo) / golden, lo + (hi - lo) / golden
    return (~outside & (pr < 0)) | (outside & (big_r((lo + hi) / 2) >= 0))


def _trace(a, r, th_cam, th, ph, p):
    g = _pose(a, r, th_cam)
    x, y, z = torch.sin(th) * torch.cos(ph), torch.sin(th) * torch.sin(ph), torch.cos(th)
    dop = 1 - g["speed"] * y
    yf, xf, zf = (-y + g["speed"]) / dop, g["neg_s"] * x / dop, g["neg_s"] * z / dop
    e = 1 / (g["alpha"] + g["w"] * g["wbar"] * yf)       # circular orbit: br = btheta = 0, bphi = 1
    pr, pt, b = e * g["ro"] * xf / g["sqrt_d"], e * g["ro"] * (-zf), e * g["wbar"] * yf
    q = pt * pt + math.cos(th_cam) ** 2 * (b * b / math.sin(th_cam) ** 2 - a * a)
    o_th, o_ph = torch.full_like(th, -1.0), torch.full_like(th, -1.0)
    if p.apriori_capture:
        idx = _escapes(g, a, r, pr, b, q).nonzero().squeeze(1)
    else:
        idx = torch.arange(th.numel(), device=th.device)
    r_cap = p.r_capture_factor * (1 + math.sqrt(1 - a * a)) if p.r_capture_factor > 0 else 0.0
    b, q = b[idx], q[idx]
    v = [torch.full_like(b, r), torch.full_like(b, th_cam), torch.zeros_like(b), pr[idx], pt[idx]]
    zz, h = torch.zeros_like(b), torch.full_like(b, math.copysign(p.h1, p.z_end))
    for n in range(p.max_steps):
        if idx.numel() == 0:
            break
        k = [_derivs(a, v, b, q)]
        scale = [v[i].abs() + (k[0][i] * h).abs() + 1e-30 for i in range(5)]
        for row in _A:
            k.append(_derivs(a, [v[i] + h * _combine(row, k, i) for i in range(5)], b, q))
        err = torch.stack([(h * _combine(_D, k, i) / scale[i]).abs() for i in range(5)]).amax(0) / p.eps
        ok = err <= 1.0
        v = [torch.where(ok, v[i] + h * _combine(_C, k, i), v[i]) for i in range(5)]
        del k, scale
        zz = torch.where(ok, zz + h, zz)
        grow = torch.where(err > 1.89e-4, 0.9 * h * err ** -0.2, 5 * h)
        h = torch.where(ok, grow, torch.minimum(0.9 * h * err ** -0.25, 0.1 * h))
        esc = zz <= p.z_end
        if p.r_escape > 0:
            esc = esc | (v[0] > p.r_escape)
        cap = ~esc & (v[0] < r_cap)
        out = ~esc & ~cap & (n + 1 >= p.max_steps)
        end = esc | out
        if bool((end | cap).any()):
            t = torch.where(esc, v[1], torch.full_like(v[1], th_cam))[end]
            f = torch.where(esc, v[2], torch.zeros_like(v[2]))[end]
            t = torch.fmod(t, 2 * PI)
            t = torch.where(t < 0, t + 2 * PI, t)
            f = torch.where(t > PI, f + PI, f)
            t = torch.where(t > PI, t - 2 * (t - PI), t)
            f = torch.remainder(f, 2 * PI)
            o_th[idx[end]], o_ph[idx[end]] = t, f
            keep = ~(end | cap)
            idx, b, q, zz, h = idx[keep], b[keep], q[keep], zz[keep], h[keep]
            v = [x[keep] for x in v]
    return o_th, o_ph
