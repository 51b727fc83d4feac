"""The workloads whose speed is watched, each through the package's public entry points.

Five kinds of call, over the sizes the package is used at:
  frame     one water frame (wt_water_displace): a projected grid, Gerstner waves, heightmap
  batch     one frame of many patches (wt_batch_set_cameras + wt_water_displace_batched)
  varyings  the vertex program's remaining outputs (wt_vertex_varyings)
  shade     the fragment stage over a fragment buffer (wt_water_shade)
  fit       the heightfield fit, one problem or a batch: gradients, or Adam iterations

Inputs are made here with torch and numpy from the seed alone; exact() restates each path
in 64 bits from the same inputs, without the package.
"""
import math
import os
import sys

import numpy as np
import torch

_PACKAGE = os.path.join(os.getcwd(), "wave-tool_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

GRAVITY = 9.81
SLAB = 2.0  # projector slab half-height, m
ADAM = dict(lr=1e-2, beta1=0.9, beta2=0.999, eps=1e-8)
SAMPLE_SCALE = 0.02
SCROLL = (0.3, 0.0)


def listed():
    return [
        # the smallest frame: a distant or preview grid, where the launch counts
        dict(name="frame_128_w16", kind="frame", n=128, waves=16, map="r32_repeat", tb=False),
        # a 256^2 grid with 4 waves, tangents and bitangents, no heightmap
        dict(name="frame_256_w4_tb", kind="frame", n=256, waves=4, map="none", tb=True),
        # the reference's own grid and wave count with an 8-bit mirrored heightmap (odd side)
        dict(name="frame_513_w4_r8", kind="frame", n=513, waves=4, map="r8_mirror", tb=False),
        # the production frame: 1024^2, 64 waves, FP32 heightmap
        dict(name="frame_1024_w64", kind="frame", n=1024, waves=64, map="r32_repeat", tb=False),
        # a few small tiles around the viewer, re-aimed every frame: launch-bound
        dict(name="batch_24_small", kind="batch", count=24, n_lo=32, n_hi=160, w_lo=4, w_hi=32),
        # 512 uneven patches (side 32-1024, 4-128 waves), re-aimed every frame
        dict(name="batch_512", kind="batch", count=512, n_lo=32, n_hi=1024, w_lo=4, w_hi=128),
        # every varying of the production frame
        dict(name="varyings_1024", kind="varyings", n=1024),
        # the fragment stage of a small window with half-size local targets, blended
        dict(name="shade_720p_blend", kind="shade", width=1280, height=720, sky=256, scale=0.5, blend=True),
        # the fragment stage of a 3840 x 2160 frame with the reference's skybox size
        dict(name="shade_4k", kind="shade", width=3840, height=2160, sky=2048, scale=1.0, blend=False),
        # a small fit, iterated: short launches one after another
        dict(name="fit_64_s8_w16", kind="fit", count=1, n_lo=64, n_hi=64, s_lo=8, s_hi=8, w_lo=16, w_hi=16, steps=10),
        # loss and gradient of one 512^2 x 16 x 32 problem, as an outer optimiser calls it
        dict(name="grad_512_s16_w32", kind="fit", count=1, n_lo=512, n_hi=512, s_lo=16, s_hi=16, w_lo=32, w_hi=32,
             steps=0),
        # 256 uneven fits (side 64-512, 8-64 waves, 4-32 snapshots) iterated together
        dict(name="fit_batch_256", kind="fit", count=256, n_lo=64, n_hi=512, s_lo=4, s_hi=32, w_lo=8, w_hi=64, steps=3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "batch", "batch", "varyings", "shade", "fit", "fit", "fit_batch"])
    if kind == "frame":
        return dict(kind="frame", n=_log_int(rng, 32, 1400), waves=_log_int(rng, 1, 128),
                    map=rng.choice(["none", "r32_repeat", "r32_mirror", "r8_repeat", "r8_mirror"]),
                    tb=rng.random() < 0.3)
    if kind == "batch":
        lo = _log_int(rng, 17, 200)
        return dict(kind="batch", count=_log_int(rng, 4, 256), n_lo=lo, n_hi=_log_int(rng, lo, 1024),
                    w_lo=rng.randint(1, 16), w_hi=rng.randint(16, 128))
    if kind == "varyings":
        return dict(kind="varyings", n=_log_int(rng, 64, 2048))
    if kind == "shade":
        width = _log_int(rng, 320, 3840)
        return dict(kind="shade", width=width, height=max(1, int(width * rng.choice([0.5625, 0.625, 0.75]))),
                    sky=rng.choice([128, 256, 512, 1024, 2048]), scale=rng.choice([0.5, 1.0]),
                    blend=rng.random() < 0.5)
    if kind == "fit":
        n, s, w = _log_int(rng, 32, 512), rng.randint(2, 32), rng.randint(4, 64)
        return dict(kind="fit", count=1, n_lo=n, n_hi=n, s_lo=s, s_hi=s, w_lo=w, w_hi=w, steps=rng.choice([0, 0, 4, 10]))
    return dict(kind="fit", count=_log_int(rng, 4, 128), n_lo=64, n_hi=_log_int(rng, 64, 512), s_lo=4,
                s_hi=rng.randint(4, 32), w_lo=8, w_hi=rng.randint(8, 64), steps=rng.choice([0, 2]))


# --------------------------------------------------------------------- shared inputs
def _dev():
    return torch.device("cuda:0")


def _wave_rows(rng, count):
    """(count, 8) float32 waves {A, w, phi, Q, Dx, Dz, phi0, 0}: L ~ U[1, 60] m, A = L / U[60, 120], direction within
    45 degrees of +x, steepness normalised by the count."""
    L = rng.uniform(1.0, 60.0, count)
    A = (L / rng.uniform(60.0, 120.0, count)).astype(np.float32)
    ang = np.radians(rng.uniform(-45.0, 45.0, count))
    w = (2.0 * math.pi / L).astype(np.float32)
    out = np.zeros((count, 8), dtype=np.float32)
    out[:, 0], out[:, 1], out[:, 2] = A, w, np.sqrt(GRAVITY * 2.0 * math.pi / L)
    out[:, 3] = rng.uniform(0.0, 1.0, count).astype(np.float32) / (w * A * np.float32(count))
    out[:, 4], out[:, 5], out[:, 6] = np.cos(ang), np.sin(ang), rng.uniform(0.0, 2.0 * math.pi, count)
    return out


def _camera(rng, far=1000.0):
    """(fov, aspect, near, far, x, y, z, yaw, pitch): 2-50 m up, looking 5-35 degrees down."""
    v = (60.0, 16.0 / 9.0, 0.1, far, rng.uniform(-100, 100), rng.uniform(2.0, 50.0), rng.uniform(-100, 100),
         rng.uniform(0.0, 360.0), rng.uniform(-35.0, -5.0))
    return tuple(float(np.float32(x)) for x in v)


def _noise(rng, size=512):
    """Tiling value noise in [0, 1], 8 octaves of smoothstep-interpolated lattices."""
    out = torch.zeros((size, size), dtype=torch.float64, device=_dev())
    total = 0.0
    centres = (torch.arange(size, device=_dev(), dtype=torch.float64) + 0.5) / size
    for o in range(8):
        cells = 4 << o
        lat = torch.from_numpy(rng.random((cells, cells))).to(_dev())
        f = centres * cells
        i0 = torch.floor(f).long() % cells
        i1 = (i0 + 1) % cells
        t = f - torch.floor(f)
        t = t * t * (3.0 - 2.0 * t)
        top, bot = lat[i0], lat[i1]
        row = top * (1 - t)[:, None] + bot * t[:, None]
        out += 0.5 ** o * (row[:, i0] * (1 - t)[None, :] + row[:, i1] * t[None, :])
        total += 0.5 ** o
    return (out / total).clamp(0.0, 1.0)


def _heightmap(rng, mode):
    """The texel tensor of a map mode (None without one)."""
    if mode == "none":
        return None
    t = _noise(rng)
    return (t * 255.0).round().to(torch.uint8) if mode.startswith("r8") else t.float()


def _map_kwargs(texels, mode):
    import wavetool_amd as wt
    if texels is None:
        return {}
    return dict(heightmap=texels, hm_format=wt.WT_TEXEL_R8_UNORM if mode.startswith("r8") else wt.WT_TEXEL_R32F,
                hm_wrap=wt.WT_WRAP_MIRRORED_REPEAT if mode.endswith("mirror") else wt.WT_WRAP_REPEAT)


def _frame_inputs(case, seed):
    rng = np.random.default_rng([seed, 11])
    cam = _camera(rng)
    r8 = case["map"].startswith("r8")
    return dict(cam=cam, waves=_wave_rows(rng, case["waves"]), texels=_heightmap(rng, case["map"]),
                time=float(rng.uniform(0.0, 3600.0)), s_d=(0.0 if case["map"] == "none" else 1.0 if r8 else 0.05),
                bounce=0.1 if r8 else 0.0, scroll=(0.0, 0.0) if r8 else SCROLL)


def _batch_sizes(case):
    """(side, waves) of every patch: side log-uniform, waves uniform. They do not depend on the seed."""
    sizes = np.random.default_rng(16)
    return [(int(round(math.exp(sizes.uniform(math.log(case["n_lo"]), math.log(case["n_hi"]))))),
             int(sizes.integers(case["w_lo"], case["w_hi"] + 1))) for _ in range(case["count"])]


def _batch_inputs(case, seed):
    rng = np.random.default_rng([seed, 12])
    specs, waves, voff, woff = [], [], 0, 0
    for n, w in _batch_sizes(case):
        specs.append(dict(n=n, w=w, cam=_camera(rng), time=float(rng.uniform(0.0, 3600.0)), voff=voff, woff=woff))
        waves.append(_wave_rows(rng, w))
        voff += n * n
        woff += w
    return dict(specs=specs, waves=np.concatenate(waves), texels=_noise(rng).float(), vertices=voff,
                step=float(rng.uniform(0.0, 2.0)))


def _surface(case, seed):
    """Positions and normals of an N^2 grid as the displacement pass leaves them (float32), and the camera."""
    rng = np.random.default_rng([seed, 13])
    n = case["n"]
    cam = _camera(rng)
    yaw = math.radians(cam[7])
    fwd, side = (math.cos(yaw), math.sin(yaw)), (-math.sin(yaw), math.cos(yaw))
    u = torch.linspace(-1, 1, n, device=_dev(), dtype=torch.float64)[None, :]
    d = 5.0 * (900.0 / 5.0) ** torch.linspace(0, 1, n, device=_dev(), dtype=torch.float64)[:, None]
    x = cam[4] + d * (fwd[0] + 1.1 * u * side[0])
    z = cam[6] + d * (fwd[1] + 1.1 * u * side[1])
    y, hx, hz = torch.zeros_like(x), torch.zeros_like(x), torch.zeros_like(x)
    for A, w, _, _, dx, dz, ph, _ in _wave_rows(rng, 12).tolist():
        th = w * (dx * x + dz * z) + ph
        y += A * torch.sin(th)
        hx += A * w * dx * torch.cos(th)
        hz += A * w * dz * torch.cos(th)
    nrm = torch.stack([-hx, torch.ones_like(hx), -hz], -1)
    nrm /= nrm.norm(dim=-1, keepdim=True)
    pos = torch.stack([x, y, z], -1)
    return dict(pos=pos.reshape(-1, 3).float().contiguous(), nrm=nrm.reshape(-1, 3).float().contiguous(), cam=cam,
                texels=_noise(rng).float(), time=float(rng.uniform(0.0, 3600.0)))


def _view_proj(cam, pitch):
    """4x4 view and projection of a camera (row, column), in double."""
    fov, aspect, zn, zf, px, py, pz, yaw, _ = cam
    cy, sy = math.cos(math.radians(yaw)), math.sin(math.radians(yaw))
    cp, sp = math.cos(math.radians(pitch)), math.sin(math.radians(pitch))
    f = np.array([cy * cp, sp, sy * cp])
    s = np.cross(f, [0.0, 1.0, 0.0])
    s /= np.linalg.norm(s)
    view = np.eye(4)
    view[0, :3], view[1, :3], view[2, :3] = s, np.cross(s, f), -f
    view[:3, 3] = -view[:3, :3] @ np.array([px, py, pz])
    t = 1.0 / math.tan(0.5 * math.radians(fov))
    proj = np.zeros((4, 4))
    proj[0, 0], proj[1, 1], proj[2, 2], proj[2, 3], proj[3, 2] = (t / aspect, t, (zf + zn) / (zn - zf),
                                                                  2.0 * zf * zn / (zn - zf), -1.0)
    return view, proj


def _shade_inputs(case, seed):
    """A fragment buffer of a rippled sea under a tilted camera, with the textures the shader samples."""
    rng = np.random.default_rng([seed, 14])
    dev, W, H = _dev(), case["width"], case["height"]
    zn, zf = 0.1, 100.0
    eye, yaw, pitch = rng.uniform(4.0, 9.0), rng.uniform(0.0, 360.0), rng.uniform(-18.0, -9.0)
    cam = (60.0, W / H, zn, zf, 0.0, eye, 0.0, yaw, pitch)
    view, proj = _view_proj(cam, pitch)
    vp = proj @ view
    right, up, fwd = view[0, :3], view[1, :3], -view[2, :3]
    th = math.tan(math.radians(30.0))
    f64 = dict(device=dev, dtype=torch.float64)
    cx = ((torch.arange(W, **f64) + 0.5) / W * 2 - 1)[None, :] * (th * W / H)
    cy = ((torch.arange(H, **f64) + 0.5) / H * 2 - 1)[:, None] * th
    d = [fwd[k] + cx * right[k] + cy * up[k] for k in range(3)]
    down = d[1] < -1e-6
    t = torch.where(down, eye / torch.where(down, -d[1], torch.ones_like(d[1])), torch.full_like(d[1], math.inf))
    along = t * sum(d[k] * fwd[k] for k in range(3))
    ok = down & (along < zf * 0.999) & (along > zn)
    px = torch.where(ok, t * d[0], torch.zeros_like(t))
    pz = torch.where(ok, t * d[2], torch.zeros_like(t))
    hx, hz, hh = torch.zeros_like(px), torch.zeros_like(px), torch.zeros_like(px)
    for _ in range(6):
        k, ang, ph, amp = rng.uniform(0.2, 1.5), rng.uniform(0, 2 * math.pi), rng.uniform(0, 2 * math.pi), rng.uniform(
            0.02, 0.08)
        arg = k * (math.cos(ang) * px + math.sin(ang) * pz) + ph
        hh += amp * torch.sin(arg)
        hx += amp * k * math.cos(ang) * torch.cos(arg)
        hz += amp * k * math.sin(ang) * torch.cos(arg)
    n = torch.stack([-hx, torch.ones_like(hx), -hz], -1)
    n /= n.norm(dim=-1, keepdim=True)
    c, s = math.cos(math.radians(yaw)), math.sin(math.radians(yaw))
    ny = torch.stack([c * n[..., 0] - s * n[..., 2], n[..., 1], s * n[..., 0] + c * n[..., 2]], -1)
    clip = [vp[r, 0] * px + vp[r, 2] * pz + vp[r, 3] for r in range(4)]
    w0 = torch.where(ok, clip[3], torch.ones_like(px))
    depth_of = lambda a: 0.5 * ((zf + zn) / (zf - zn) - 2 * zf * zn / ((zf - zn) * a)) + 0.5  # noqa: E731
    rec = torch.cat([n, torch.stack([-px, eye - hh, -pz], -1), ny, torch.stack([clip[0] / w0, clip[1] / w0], -1),
                     depth_of(torch.where(ok, along, torch.ones_like(along)))[..., None]], -1)
    frags = torch.where(ok[..., None], rec, torch.zeros_like(rec)).float().contiguous()
    bed = 3.5 + 2.5 * torch.sin(0.05 * px + 0.3) * torch.cos(0.07 * pz)
    at_bed = along * (eye + bed) / eye
    depth = torch.where(down & (at_bed < zf), depth_of(torch.where(down, at_bed, torch.ones_like(t))),
                        torch.ones_like(t)).float().contiguous()
    lw, lh = max(1, round(W * case["scale"])), max(1, round(H * case["scale"]))

    def image(h, w, masked):
        gy = torch.linspace(0, 1, h, **f64)[:, None]
        gx = torch.linspace(0, 1, w, **f64)[None, :]
        ch = []
        for _ in range(3):
            a, b, p, q = rng.uniform(3, 12), rng.uniform(3, 12), rng.uniform(0, 6), rng.uniform(0, 6)
            ch.append(0.5 + 0.3 * torch.sin(a * gx + p) * torch.cos(b * gy + q) + 0.1 * torch.sin(5 * a * gx + 7 * b * gy))
        ch.append((ch[0] > 0.5).double() if masked else torch.ones_like(ch[0]))
        return (torch.stack(ch, -1) * 255.0).round().to(torch.uint8).contiguous()

    refl, refr = image(lh, lw, True), image(lh, lw, False)
    sky = torch.stack([image(case["sky"], case["sky"], False) for _ in range(6)]).contiguous()
    sun = rng.uniform(0.6, 2.4)
    k = max(0.0, math.sin(sun))
    uniforms = {"fogColourFarAtCurrentTime": [k, k, k, 0.1], "fogDepthRadiusFar": 1.0, "fogDepthRadiusNear": 0.0,
                "softEdgesDeltaDepthThreshold": 0.05, "sunPosition": [math.cos(sun), math.sin(sun), 0.0],
                "sunShininess": 50.0, "sunStrength": 1.0, "tintDeltaDepthThreshold": 0.1,
                "viewportWidthHeight": [float(W), float(H)], "waterClarity": 0.3, "zFar": zf, "zNear": zn}
    colour = torch.from_numpy(rng.random((1, 1, 4)).astype(np.float32)).to(dev).expand(H, W, 4).contiguous()
    return dict(uniforms=uniforms, frags=frags, cover=ok.to(torch.uint8).contiguous(), depth=depth, refl=refl, refr=refr,
                sky=sky, colour=colour)


def _fit_specs(case, seed):
    """Sizes and waves of every problem of a fit case. The sizes do not depend on the seed."""
    sizes = np.random.default_rng(17)
    rng = np.random.default_rng([seed, 15])
    out, off = [], 0
    for i in range(case["count"]):
        n = int(round(math.exp(sizes.uniform(math.log(case["n_lo"]), math.log(case["n_hi"])))))
        W, S = (int(sizes.integers(case[k + "_lo"], case[k + "_hi"] + 1)) for k in ("w", "s"))
        r = _wave_rows(rng, W).astype(np.float64)
        hidden = np.stack([r[:, 0], 2.0 * math.pi / r[:, 1], np.arctan2(r[:, 5], r[:, 4]), r[:, 3], r[:, 6]], 1)
        init = hidden * rng.uniform(0.8, 1.2, hidden.shape)
        init[:, 2] = hidden[:, 2] + np.radians(rng.uniform(-15.0, 15.0, W))
        out.append(dict(n=n, S=S, W=W, hidden=hidden, init=init.astype(np.float32), off=off, x0=-0.25 * (n - 1), seed=i))
        off += W
    return out


def _displacement(sp, params, t0=0.0, dt=0.25, spacing=0.5):
    """[S][n*n][3] displacement of wave parameters (W, 5) in double; differentiable."""
    A, L, al, Q, ph = (params[:, k] for k in range(5))
    i = torch.arange(sp["n"] ** 2, device=params.device)
    x = sp["x0"] + (i % sp["n"]).double() * spacing
    z = sp["x0"] + (i // sp["n"]).double() * spacing
    w = 2.0 * math.pi / L
    om = torch.sqrt(GRAVITY * w)
    dx, dz = torch.cos(al), torch.sin(al)
    th = x[:, None] * (w * dx)[None, :] + z[:, None] * (w * dz)[None, :] + ph[None, :]
    E = torch.cat([torch.cos(th), torch.sin(th)], 1)  # points x 2W, at time 0
    t = t0 + dt * torch.arange(sp["S"], device=params.device, dtype=torch.float64)
    c, s = torch.cos(om[:, None] * t), torch.sin(om[:, None] * t)  # W x S
    qx, qz, a = (Q * A * dx)[:, None], (Q * A * dz)[:, None], A[:, None]
    B = torch.cat([torch.stack([qx * c, a * s, qz * c], -1), torch.stack([-qx * s, a * c, -qz * s], -1)], 0)
    return (E @ B.reshape(2 * sp["W"], -1)).reshape(-1, sp["S"], 3).transpose(0, 1)


def _fit_target(sp, seed):
    """The hidden waves' displacement plus N(0, 0.01 m) on every component, float32 [S][n*n][3]."""
    g = torch.Generator(device=_dev())
    g.manual_seed((int(seed) * 1009 + sp["seed"]) & 0x7FFFFFFF)
    with torch.no_grad():
        d = _displacement(sp, torch.from_numpy(sp["hidden"]).to(_dev())).float()
    return d.contiguous() + 0.01 * torch.randn(d.shape, generator=g, device=_dev(), dtype=torch.float32)


# --------------------------------------------------------------------- the calls
def prepare(case, seed):
    import wavetool_amd as wt
    dev, kind = _dev(), case["kind"]
    ctx = wt.Context()
    if kind == "frame":
        q = _frame_inputs(case, seed)
        n = case["n"]
        params = wt.water_params(wt.projector_corners(q["cam"], SLAB), q["cam"][4:7], n, q["time"], SAMPLE_SCALE,
                                 q["s_d"], q["bounce"], q["scroll"])
        out = [torch.zeros(n * n * 3, device=dev) for _ in range(4 if case["tb"] else 2)]
        return dict(kind=kind, ctx=ctx, params=params, waves=torch.from_numpy(q["waves"]).to(dev), out=out,
                    map=_map_kwargs(q["texels"], case["map"]))
    if kind == "batch":
        q = _batch_inputs(case, seed)
        patches = [wt.patch(np.eye(4), s["cam"][4:7], s["n"], s["woff"], s["w"], s["voff"], s["time"], SAMPLE_SCALE,
                            0.05, 0.0, SCROLL) for s in q["specs"]]
        count = len(patches)
        return dict(kind=kind, ctx=ctx, batch=wt.Batch(ctx, patches), waves=torch.from_numpy(q["waves"]).to(dev),
                    cams=torch.from_numpy(wt.camera_rows([s["cam"] for s in q["specs"]])).to(dev),
                    amps=torch.full((count,), SLAB, device=dev), status=torch.zeros(count, dtype=torch.int32, device=dev),
                    map=q["texels"], pos=torch.zeros(q["vertices"] * 3, device=dev),
                    nrm=torch.zeros(q["vertices"] * 3, device=dev), step=q["step"])
    if kind == "varyings":
        q = _surface(case, seed)
        v = case["n"] ** 2
        view, proj = _view_proj(q["cam"], q["cam"][8])
        params = wt.water_params(np.zeros((4, 4)), q["cam"][4:7], case["n"], q["time"], SAMPLE_SCALE, 0.05, 0.0, SCROLL)
        outs = {k: torch.zeros(v * m, device=dev) for k, m in (("clip", 4), ("ndc0", 2), ("view", 3), ("nview", 3),
                                                             ("sample", 1))}
        return dict(kind=kind, ctx=ctx, params=params, vp=proj @ view, vy=_view_proj(q["cam"], 0.0)[0], pos=q["pos"],
                    nrm=q["nrm"], map=q["texels"], count=v, outs=outs)
    if kind == "shade":
        q = _shade_inputs(case, seed)
        q.update(kind=kind, ctx=ctx, blend=case["blend"], uniforms=wt.shade_params(q["uniforms"]))
        return q
    specs = _fit_specs(case, seed)
    params = torch.from_numpy(np.concatenate([s["init"] for s in specs])).to(dev)
    targets = [_fit_target(s, seed) for s in specs]
    problems = [wt.fit_problem(s["n"], s["S"], s["W"], 0.5, s["x0"], s["x0"], 0.0, 0.25, t,
                               params[s["off"]:s["off"] + s["W"]]) for s, t in zip(specs, targets)]
    torch.cuda.synchronize()
    return dict(kind="fit", ctx=ctx, fit=wt.Fit(ctx, problems), params=params, targets=targets, steps=case["steps"],
                grad=torch.zeros(params.numel(), device=dev), losses=torch.zeros(len(specs), device=dev))


def run(state):
    kind = state["kind"]
    if kind == "frame":
        out = state["out"]
        state["ctx"].displace(state["params"], state["waves"], *out, **state["map"])
        return out
    if kind == "batch":
        state["batch"].set_cameras(state["cams"], state["amps"], state["status"])
        state["batch"].displace(state["waves"], state["pos"], state["nrm"], heightmap=state["map"],
                                time_offset=state["step"])
        return dict(pos=state["pos"], nrm=state["nrm"], status=state["status"])
    if kind == "varyings":
        state["ctx"].varyings(state["params"], state["vp"], state["vy"], state["pos"], state["nrm"], state["count"],
                              heightmap=state["map"], **state["outs"])
        return state["outs"]
    if kind == "shade":
        state["ctx"].shade(state["uniforms"], state["depth"], state["refl"], state["refr"], state["sky"], state["frags"],
                           state["colour"], coverage=state["cover"], blend=state["blend"])
        return state["colour"]
    if state["steps"]:
        state["fit"].iterate(state["steps"], losses=state["losses"], **ADAM)
        return dict(params=state["params"], losses=state["losses"])
    state["fit"].loss_grad(state["grad"], state["losses"])
    return dict(grad=state["grad"], losses=state["losses"])


def work(case):
    """FLOP: 26 per vertex-wave (phase 5, sine and cosine 2, position 7, partial derivatives 12); a fit: 20 per
    vertex-wave-snapshot (sine and cosine 2, displacement 6, the residual's products with both 12), the Adam update of a
    few hundred parameters aside. Bytes: every input once, every output once."""
    kind = case["kind"]
    texels = 512 * 512 * 4
    if kind == "frame":
        v = case["n"] ** 2
        t = 0 if case["map"] == "none" else texels // 4 if case["map"].startswith("r8") else texels
        return dict(bytes=v * (48 if case["tb"] else 24) + case["waves"] * 32 + t, flops=26 * v * case["waves"])
    if kind == "batch":
        sizes = _batch_sizes(case)
        return dict(bytes=texels + sum(n * n * 24 + w * 32 + 40 for n, w in sizes), flops=26 * sum(n * n * w for n, w in sizes))
    if kind == "varyings":
        return dict(bytes=case["n"] ** 2 * 76 + texels, flops=case["n"] ** 2 * 60)
    if kind == "shade":
        # about 63% of the frame is sea: 80 B a covered pixel (+ 16 to blend), the coverage byte of every pixel
        v = case["width"] * case["height"]
        return dict(bytes=v * (1 + 0.63 * (96 if case["blend"] else 80)), flops=0.63 * v * 300)
    sizes = _fit_specs(case, 0)
    passes = max(1, case["steps"])
    return dict(bytes=passes * sum(s["n"] ** 2 * s["S"] * 12 + s["W"] * 40 for s in sizes),
                flops=passes * 20 * sum(s["n"] ** 2 * s["S"] * s["W"] for s in sizes))


# --------------------------------------------------------------------- in 64 bits
def _corners(cam, amp):
    """The projected grid's corners (BL, TL, BR, TR) of a camera, and a status, in double: the padded frustum's points
    inside |y| <= amp seen from a projector above the slab."""
    fov, aspect, zn, zf, px, py, pz, yaw, pitch = cam
    pos = np.array([px, py, pz])

    def look(p, yaw_, pitch_):
        c = (fov, aspect, zn, zf, p[0], p[1], p[2], yaw_, pitch_)
        return _view_proj(c, pitch_)

    def on_plane(a, b, y):
        d = (b - a) / np.linalg.norm(b - a)
        return None if d[1] == 0.0 else a + d * ((y - a[1]) / d[1])

    pitch = min(89.0, max(-89.0, pitch))
    view, proj = look(pos, yaw, pitch)
    inv = np.linalg.inv(proj @ view)
    fc = []
    for i in range(8):
        q = inv @ np.array([1.2 * (1 if i & 4 else -1), 1.2 * (1 if i & 2 else -1), 1.0 if i & 1 else -1.0, 1.0])
        fc.append(q[:3] / q[3])
    f = -view[2, :3]
    low = amp + 1.0
    pj = pos + (np.array([0.0, low - 2 * py if py < 0 else low - py, 0.0]) if py < low else 0.0)
    fy = f.copy()
    if abs(fy[1]) < 0.001:
        fy[1] = math.copysign(0.001, fy[1])
    ray = fy if (fy[1] < 0) != (py < 0) else fy * np.array([1.0, -1.0, 1.0])
    aim1 = on_plane(pos, pos + ray, 0.0)
    aim2 = (pos + f) * np.array([1.0, 0.0, 1.0])
    a = abs(fy[1])
    nf = (aim2 * (1 - a) + aim1 * a) - pj
    nf /= np.linalg.norm(nf)
    flat = nf * np.array([1.0, 0.0, 1.0])
    flat /= np.linalg.norm(flat)
    pview, pproj = look(pj, yaw, -math.degrees(math.acos(min(1.0, max(-1.0, float(nf @ flat))))))
    pvp = pproj @ pview
    pts = []
    for i, j in ((0, 1), (0, 2), (0, 4), (1, 3), (1, 5), (2, 3), (2, 6), (3, 7), (4, 5), (4, 6), (5, 7), (6, 7)):
        lo, hi = min(fc[i][1], fc[j][1]), max(fc[i][1], fc[j][1])
        for y in (amp, -amp):
            if lo <= y <= hi:
                hit = on_plane(fc[i], fc[j], y)
                if hit is not None:
                    pts.append(hit)
    pts += [p for p in fc if -amp <= p[1] <= amp]
    if not pts:
        return None, 2
    lo = hi = None
    for p in pts:  # as the reference does: a point that lowers the minimum never raises the maximum
        q = pvp @ np.array([p[0], 0.0, p[2], 1.0])
        v = q[:2] / q[3]
        if lo is None:
            lo, hi = v.copy(), v.copy()
            continue
        for k in range(2):
            if v[k] < lo[k]:
                lo[k] = v[k]
            elif v[k] > hi[k]:
                hi[k] = v[k]
    back = np.linalg.inv(proj @ pview)
    out = np.ones((4, 4))
    for i in range(4):
        x, y = lo[0] + (i >> 1) * (hi[0] - lo[0]), lo[1] + (i & 1) * (hi[1] - lo[1])
        n, r = back @ np.array([x, y, -1.0, 1.0]), back @ np.array([x, y, 1.0, 1.0])
        out[i, :3] = on_plane(n[:3] / n[3], r[:3] / r[3], 0.0)
    return out, 0


def _tap(texels, mirror, s, t):
    """Bilinear value and its derivatives by (s, t) of a wrapped texture, in double."""
    h, w = texels.shape
    tex = texels.double() / 255.0 if texels.dtype == torch.uint8 else texels.double()

    def wrap(i, n):
        if not mirror:
            return i % n
        i = i % (2 * n)
        return torch.minimum(i, 2 * n - 1 - i)

    u, v = s * w - 0.5, t * h - 0.5
    fu, fv = torch.floor(u), torch.floor(v)
    a, b = u - fu, v - fv
    i, j = fu.long(), fv.long()
    i0, i1, j0, j1 = wrap(i, w), wrap(i + 1, w), wrap(j, h), wrap(j + 1, h)
    t00, t10, t01, t11 = tex[j0, i0], tex[j0, i1], tex[j1, i0], tex[j1, i1]
    lo, hi = t00 + a * (t10 - t00), t01 + a * (t11 - t01)
    ds = w * ((1 - b) * (t10 - t00) + b * (t11 - t01))
    dt = h * ((1 - a) * (t01 - t00) + a * (t11 - t10))
    return lo + b * (hi - lo), ds, dt


def _vertices(corners, cam_pos, n, time, waves, texels, mirror, s_d, bounce, scroll, tb):
    """Position, normal (and tangent, bitangent) of every vertex, in double, on the GPU."""
    dev = _dev()
    c = torch.from_numpy(corners).to(dev)
    waves = torch.from_numpy(waves.astype(np.float64)).to(dev)
    outs = [torch.empty((n * n, 3), dtype=torch.float64, device=dev) for _ in range(4 if tb else 2)]
    rows = max(1, (1 << 23) // max(1, n * len(waves)))
    s_h = float(np.float32(SAMPLE_SCALE))
    s_d, bounce = float(np.float32(s_d)), float(np.float32(bounce))
    sx, sz = float(np.float32(scroll[0])), float(np.float32(scroll[1]))
    for r0 in range(0, n, rows):
        r1 = min(n, r0 + rows)
        u = (torch.arange(n, device=dev, dtype=torch.float64) / (n - 1))[None, :]
        v = (torch.arange(r0, r1, device=dev, dtype=torch.float64) / (n - 1))[:, None]
        x, z = ((c[0, k] + u * (c[2, k] - c[0, k])) * (1 - v) + (c[1, k] + u * (c[3, k] - c[1, k])) * v for k in (0, 2))
        x, z = x.reshape(-1), z.reshape(-1)
        A, w, phi, Q, dx, dz, ph0 = (waves[:, k] for k in range(7))
        th = x[:, None] * (w * dx) + z[:, None] * (w * dz) + (phi * time + ph0)
        co, si = torch.cos(th), torch.sin(th)
        X, Z, Y = co @ (Q * A * dx), co @ (Q * A * dz), si @ A
        tx, ty, tz = 1 - si @ (Q * A * w * dx * dx), co @ (A * w * dx), -(si @ (Q * A * w * dx * dz))
        bx, by, bz = tz, co @ (A * w * dz), 1 - si @ (Q * A * w * dz * dz)
        px, pz, py = x + X, z + Z, Y
        if texels is not None:
            val, ds, dt = _tap(texels, mirror, s_h * (px - sx * time), -s_h * (pz - sz * time))
            py = py + 2 * s_d * (val - 0.5)
            hx, hz = 2 * s_d * s_h * ds, -2 * s_d * s_h * dt
            ty, by = ty + hx * tx + hz * tz, by + hx * bx + hz * bz
        py = py + bounce
        P, T, B = torch.stack([px, py, pz], 1), torch.stack([tx, ty, tz], 1), torch.stack([bx, by, bz], 1)
        N = torch.linalg.cross(B, T)
        N = N / N.norm(dim=1, keepdim=True)
        V = torch.tensor([float(q) for q in cam_pos], device=dev, dtype=torch.float64)[None, :] - P
        N = torch.where((N * V).sum(1, keepdim=True) < 0, -N, N)
        for o, val in zip(outs, (P, N, T / T.norm(dim=1, keepdim=True), B / B.norm(dim=1, keepdim=True))):
            o[r0 * n:r1 * n] = val
    return [o.reshape(-1) for o in outs]


def _rgba(tex, s, t):
    """GL_LINEAR, CLAMP_TO_EDGE of an RGBA8 image, in double."""
    h, w = tex.shape[:2]
    u, v = s * w - 0.5, t * h - 0.5
    fu, fv = torch.floor(u), torch.floor(v)
    a, b = (u - fu)[..., None], (v - fv)[..., None]
    i0, i1 = fu.long().clamp(0, w - 1), (fu.long() + 1).clamp(0, w - 1)
    j0, j1 = fv.long().clamp(0, h - 1), (fv.long() + 1).clamp(0, h - 1)
    g = lambda j, i: tex[j, i].double() / 255.0  # noqa: E731
    return (g(j0, i0) * (1 - a) + g(j0, i1) * a) * (1 - b) + (g(j1, i0) * (1 - a) + g(j1, i1) * a) * b


def _shaded(case, q):
    """The fragment colours over the destination, in double."""
    un, f = q["uniforms"], q["frags"].double()
    f32 = lambda v: float(np.float32(v))  # noqa: E731
    H, W = f.shape[:2]
    dev = f.device
    out = q["colour"].double().clone()
    sel = q["cover"].bool()
    f = f[sel]
    rows, cols = torch.nonzero(sel, as_tuple=True)
    uvx, uvy = (cols.double() + 0.5) / W, (rows.double() + 0.5) / H
    zf, zn = f32(un["zFar"]), f32(un["zNear"])
    lin = lambda d: zn * d / (zf - d * (zf - zn))  # noqa: E731
    back = lin(q["depth"].double()[rows, cols])
    n, view, ny, ndc = f[:, 0:3], f[:, 3:6], f[:, 6:9], f[:, 9:11]
    length = view.norm(dim=1)
    clamped = (length / zf).clamp(0, 1)
    in_front = (back <= f32(0.999)).double()
    delta = (back - lin(f[:, 11])).clamp(0, 1)
    v = view / length[:, None]
    nd = (n * v).sum(1)
    r = -v + 2 * nd[:, None] * n
    ax = r.abs()
    out_sky = torch.zeros((len(f), 4), device=dev, dtype=torch.float64)
    x_major = (ax[:, 0] >= ax[:, 1]) & (ax[:, 0] >= ax[:, 2])
    y_major = ~x_major & (ax[:, 1] >= ax[:, 2])
    for k, major, sc, tc in ((0, x_major, lambda g, s: -s * g[:, 2], lambda g, s: -g[:, 1]),
                             (1, y_major, lambda g, s: g[:, 0], lambda g, s: s * g[:, 2]),
                             (2, ~x_major & ~y_major, lambda g, s: s * g[:, 0], lambda g, s: -g[:, 1])):
        for side, face in ((1.0, 2 * k), (-1.0, 2 * k + 1)):
            m = major & ((r[:, k] >= 0) == (side > 0))
            g = r[m]
            ma = g[:, k].abs()
            out_sky[m] = _rgba(q["sky"][face], 0.5 * (sc(g, side) / ma + 1), 0.5 * (tc(g, side) / ma + 1))
    sun_dir = torch.tensor([f32(s) for s in un["sunPosition"]], device=dev, dtype=torch.float64)
    sun = f32(un["sunStrength"]) * (r @ sun_dir).clamp(0, 1) ** f32(un["sunShininess"])
    fresnel = 0.02 + 0.98 * (1 - nd) ** 5
    dist = 0.1 * (1 - clamped)
    yx, yy = (uv * (1 - dist) + (ndc[:, k] + 1) * 0.5 * dist for k, uv in ((0, uvx), (1, uvy)))
    lrefl = _rgba(q["refl"], (yx + dist * ny[:, 0]).clamp(0, 1), (yy - dist * ny[:, 2]).clamp(0, 1))
    lrefr = _rgba(q["refr"], (yx - dist * ny[:, 0]).clamp(0, 1), (yy + dist * ny[:, 2]).clamp(0, 1))
    tint = (in_front * (1 - (delta / f32(un["tintDeltaDepthThreshold"])).clamp(0, 1)))[:, None]
    deep = torch.tensor([0.0, 0.341, 0.482], device=dev, dtype=torch.float64)
    shallow = torch.tensor([0.3, 0.941, 0.903], device=dev, dtype=torch.float64)
    tinted = (deep * (1 - tint) + shallow * tint) * min(1.0, max(0.0, float(sun_dir[1])))
    k = (f32(un["waterClarity"]) * lrefr[:, 3] * (1 - delta))[:, None]
    through = tinted * (1 - k) + lrefr[:, :3] * k
    mirror = (out_sky[:, :3] + sun[:, None]) * (1 - lrefl[:, 3:]) + lrefl[:, :3] * lrefl[:, 3:]
    colour = through * (1 - fresnel[:, None]) + mirror * fresnel[:, None]
    alpha = 1 - in_front * (1 - (delta / f32(un["softEdgesDeltaDepthThreshold"])).clamp(0, 1))
    fog = [f32(x) for x in un["fogColourFarAtCurrentTime"]]
    fa = (fog[3] * clamped)[:, None]
    colour = colour * (1 - fa) + torch.tensor(fog[:3], device=dev, dtype=torch.float64) * fa
    res = torch.cat([colour, alpha[:, None]], 1)
    out[sel] = res * alpha[:, None] + out[sel] * (1 - alpha[:, None]) if case["blend"] else res
    return out


def _fit_exact(case, seed):
    specs = _fit_specs(case, seed)
    b1, b2, lr, eps = (float(np.float32(ADAM[k])) for k in ("beta1", "beta2", "lr", "eps"))
    every, losses = [], []
    for sp in specs:
        target = _fit_target(sp, seed)
        p = torch.from_numpy(sp["init"]).to(_dev()).double()
        m, v = torch.zeros_like(p), torch.zeros_like(p)
        for step in range(1, max(1, case["steps"]) + 1):
            q = p.clone().requires_grad_(True)
            r = _displacement(sp, q) - target
            loss = 0.5 * r.square().sum() / (sp["S"] * sp["n"] ** 2)
            loss.backward()
            g = q.grad
            if case["steps"]:
                m, v = b1 * m + (1 - b1) * g, b2 * v + (1 - b2) * g * g
                p = p - lr * (m / (1 - b1 ** step)) / ((v / (1 - b2 ** step)).sqrt() + eps)
                p[:, 1].clamp_(min=1e-3)
        every.append(p if case["steps"] else g)
        losses.append(loss.detach())
    out = torch.cat(every)
    return dict(params=out, losses=torch.stack(losses)) if case["steps"] else dict(grad=out.reshape(-1),
                                                                                 losses=torch.stack(losses))


def exact(case, seed):
    kind = case["kind"]
    if kind == "frame":
        q = _frame_inputs(case, seed)
        return _vertices(_corners(q["cam"], SLAB)[0], q["cam"][4:7], case["n"], q["time"], q["waves"], q["texels"],
                         case["map"].endswith("mirror"), q["s_d"], q["bounce"], q["scroll"], case["tb"])
    if kind == "batch":
        q = _batch_inputs(case, seed)
        pos = torch.zeros(q["vertices"] * 3, dtype=torch.float64, device=_dev())
        nrm = torch.zeros_like(pos)
        status = []
        for s in q["specs"]:
            corners, st = _corners(s["cam"], SLAB)
            status.append(st)
            if st == 0:
                at = slice(3 * s["voff"], 3 * (s["voff"] + s["n"] ** 2))
                pos[at], nrm[at] = _vertices(corners, s["cam"][4:7], s["n"], s["time"] + q["step"],
                                             q["waves"][s["woff"]:s["woff"] + s["w"]], q["texels"], False, 0.05, 0.0,
                                             SCROLL, False)
        return dict(pos=pos, nrm=nrm, status=torch.tensor(status, dtype=torch.int32))
    if kind == "varyings":
        q = _surface(case, seed)
        f32 = lambda m: torch.from_numpy(np.asarray(m, dtype=np.float32)).double().to(_dev())  # noqa: E731
        view, proj = _view_proj(q["cam"], q["cam"][8])
        vp, vy = f32(proj @ view), f32(_view_proj(q["cam"], 0.0)[0])
        P, N = q["pos"].double(), q["nrm"].double()
        one = torch.ones_like(P[:, :1])
        clip = torch.cat([P, one], 1) @ vp.T
        flat = torch.stack([P[:, 0], torch.zeros_like(P[:, 0]), P[:, 2], one[:, 0]], 1) @ vp.T
        nv = (N @ vy[:3, :3].T)
        s_h, sx = float(np.float32(SAMPLE_SCALE)), float(np.float32(SCROLL[0]))
        val = _tap(q["texels"], False, s_h * (P[:, 0] - sx * q["time"]), -s_h * P[:, 2])[0]
        cam = f32(np.array(q["cam"][4:7]))
        return dict(clip=clip.reshape(-1), ndc0=(flat[:, :2] / flat[:, 3:]).reshape(-1), view=(cam - P).reshape(-1),
                    nview=(nv / nv.norm(dim=1, keepdim=True)).reshape(-1), sample=val)
    if kind == "shade":
        return _shaded(case, _shade_inputs(case, seed))
    return _fit_exact(case, seed)
