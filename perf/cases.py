"""The work that a user of this renderer has it do, as measurable cases.

Each case is one pass through the public renderers: a training pass (the
maps, then the gradients of every parameter for the gradient images that a
program's image loss hands back) or a rendering pass (no gradients). They
span the sizes of this repository's workloads, from a 64x64 frame of a
thousand surfels, where launches and host time decide, to a million surfels
at 1080p and 32 views at once.

Scenes follow the distributions of ``workloads.py`` (means in a frustum box
or in Gaussian clusters, log-uniform scales, opacities U(0.1, 0.9), SH or
direct colours, SIREN weights), but for the orientations: surfels face
the viewing ray within an angle (cosine at least `tilt`), either face up, as
the visible surfels of fitted surfaces do, rather than uniformly over the
sphere, where a few edge-on surfels dominate every gradient with rounding
noise.
"""

from __future__ import annotations

import contextlib
import math

import torch

from diff_gabor_splatting_amd import fixed_capacity, rasterize_gabors, rasterize_neural_gabors

PARAMETERS = ("means", "quaternions", "scales", "opacities")
CLASSIC = ("colors", "secondary_colors", "frequency_weights", "frequency_magnitudes", "phases")
NEURAL = ("input_weights", "input_biases", "output_weights", "output_biases")
NEURAL_SHAPES = ((6, 5), (6,), (3, 6), (3,))
CAMERAS = ("view_matrices", "intrinsics", "backgrounds")
MAP_CHANNELS = 9
BOXES = {  # means: half width in x and y, nearest and farthest depth
    "near": (1.0, 2.0, 4.0),      # a small object in front of the camera
    "room": (3.0, 2.0, 8.0),      # a room-sized frustum
    "clusters": (5.0, 2.0, 12.0),  # 64 Gaussian clusters: heavy overlap
    "ring": (2.0, 3.0, 7.0),      # cameras on an arc around the box's centre
}
LIMIT = 1.2e11  # estimated floating-point operations that a drawn case may take


def _case(name, **options):
    case = dict(name=name, train=True, neural=False, scenes=1, cameras=1, n=1024, width=64,
                height=64, sh=-1, packed=False, validate=True, box="room", scale_low=0.02,
                scale_high=0.2, tilt=0.4, focal=0.88, maps="all", backgrounds=False,
                poses=False, capacity=0)
    case.update(options)
    return case


def listed():
    return [
        # A preview or a unit-sized fit: the smallest frame that the renderer
        # is called on, without gradients. Latency and launches count.
        _case("render_small", train=False, sh=0, box="near", focal=1.25),
        # The same frame in an optimisation loop (texture fits, debugging runs).
        _case("train_small", sh=0, box="near", focal=1.25, validate=False),
        # A few views of one small scene per step, direct colours, checked
        # inputs (the defaults): the usual multi-view fit at low resolution.
        _case("train_views", cameras=4, n=10_000, width=256, height=256, maps="all",
              scale_low=0.01, scale_high=0.06, box="near", focal=1.1),
        # The neural renderer's counterpart.
        _case("train_views_neural", neural=True, cameras=4, n=10_000, width=256, height=256,
              scale_low=0.01, scale_high=0.06, box="near", focal=1.1),
        # Rendering frames in a loop that must not wait for the GPU.
        _case("render_stream", train=False, n=30_000, width=640, height=480, packed=False,
              validate=False, scale_low=0.02, scale_high=0.1, capacity=4_000_000),
        # Ragged sizes and every option together: packed rows, SH degree 2, a
        # coloured background, camera refinement.
        _case("train_ragged", cameras=3, n=33_333, width=517, height=389, sh=2, packed=True,
              backgrounds=True, poses=True, scale_low=0.02, scale_high=0.1),
        # A full-resolution training step of a mid-sized scene, rgb, alpha and
        # depth supervised.
        _case("train_frame", n=100_000, width=1024, height=768, sh=3, validate=False,
              maps="depth"),
        # Neural surfels at 800x800, trained and rendered.
        _case("train_neural", neural=True, n=100_000, width=800, height=800, validate=False,
              focal=1.125),
        _case("render_neural", train=False, neural=True, n=100_000, width=800, height=800,
              focal=1.125),
        # A batch of scenes and cameras in one packed call.
        _case("train_batch", scenes=8, cameras=4, n=50_000, width=512, height=512, sh=3,
              packed=True, validate=False, box="ring", tilt=0.8, focal=1.17),
        # A large scene at 1080p: its training step and a rendered frame.
        _case("train_large", n=1_000_000, width=1920, height=1080, sh=3, validate=False,
              box="clusters", scale_low=0.005, scale_high=0.1, focal=0.78),
        _case("render_large", train=False, n=1_000_000, width=1920, height=1080, sh=3,
              box="clusters", scale_low=0.005, scale_high=0.1, focal=0.78),
    ]


def _log(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def draw(rng):
    """One more case: any size between the smallest and the largest listed
    one, odd sizes among them, with any of the options."""
    while True:
        neural = rng.random() < 0.35
        cameras = rng.choice((1, 1, 1, 2, 3, 4))
        box = rng.choice(("near", "room", "room", "clusters", "ring"))
        most = {"near": 30_000, "ring": 100_000}.get(box, 200_000 if neural else 1_000_000)
        n = int(_log(rng, 900, most))
        # Surfels shrink as their number grows, as fitted scenes' do.
        middle = rng.uniform(0.5, 1.1) * 0.06 * BOXES[box][0] / 3 * math.sqrt(1e5 / n)
        middle = min(max(middle, 0.008), 0.25)
        case = _case("", train=rng.random() < 0.7, neural=neural,
                     scenes=rng.choice((1, 1, 1, 2)), cameras=cameras, n=n,
                     width=int(_log(rng, 48, 1920)), height=int(_log(rng, 48, 1080)),
                     sh=-1 if neural else rng.choice((-1, 0, 1, 2, 3)),
                     packed=rng.random() < 0.4, validate=rng.random() < 0.5, box=box,
                     scale_low=middle / 3, scale_high=middle * 3,
                     tilt=0.8 if box == "ring" else 0.4, focal=rng.uniform(0.8, 1.25),
                     maps=rng.choice(("all", "all", "depth", "rgb")),
                     backgrounds=rng.random() < 0.5, poses=rng.random() < 0.2)
        del case["name"]
        if work(case)["flops"] <= LIMIT:
            return case


# Inputs ---------------------------------------------------------------------

def _inputs(case, seed, device):
    """The call's tensors and the gradient images, from the seed alone."""
    g = torch.Generator(device=device).manual_seed(1_000_003 * seed + 17)

    def uniform(shape, low, high):
        return torch.rand(shape, generator=g, device=device) * (high - low) + low

    S, C, N = case["scenes"], case["cameras"], case["n"]
    W, H = case["width"], case["height"]
    half, near, far = BOXES[case["box"]]
    if case["box"] == "clusters":
        centres = torch.cat([uniform((64, 2), -half, half), uniform((64, 1), near, far)], -1)
        which = torch.randint(0, 64, (S, N), generator=g, device=device)
        means = centres[which] + 0.3 * torch.randn((S, N, 3), generator=g, device=device)
    else:
        means = torch.cat([uniform((S, N, 2), -half, half), uniform((S, N, 1), near, far)], -1)
    # Orientation: spin in the surfel's plane, tilt away from the ray through
    # the surfel's centre from the origin (the first camera's, where it does
    # not turn), half of them turned over.
    spin, axis = uniform((S, N), 0, 2 * math.pi), uniform((S, N), 0, 2 * math.pi)
    tilt = torch.acos(uniform((S, N), case["tilt"], 1.0))
    tilt = torch.where(uniform((S, N), 0, 1) < 0.5, tilt, math.pi - tilt)
    c, s = torch.cos(tilt / 2), torch.sin(tilt / 2)
    w, x = c * torch.cos(spin / 2), s * torch.cos(axis - spin / 2)
    y, z = s * torch.sin(axis - spin / 2), c * torch.sin(spin / 2)
    ray = means / means.norm(dim=-1, keepdim=True)
    a, b, d = 1 + ray[..., 2], -ray[..., 1], ray[..., 0]  # turns +z onto the ray
    quats = torch.stack([a * w - b * x - d * y, a * x + b * w + d * z, a * y - b * z + d * w,
                         a * z + b * y - d * x], -1)
    values = {
        "means": means,
        "quaternions": quats / quats.norm(dim=-1, keepdim=True),
        "scales": torch.exp(uniform((S, N, 2), math.log(case["scale_low"]),
                                    math.log(case["scale_high"]))),
        "opacities": uniform((S, N), 0.1, 0.9),
    }
    if case["neural"]:
        values["input_weights"] = uniform((S, N, 6, 5), -0.2, 0.2)
        values["input_biases"] = uniform((S, N, 6), -0.02, 0.02)
        values["output_weights"] = uniform((S, N, 3, 6), -0.4, 0.4)
        values["output_biases"] = uniform((S, N, 3), -0.5, 0.5)
    else:
        colour = (3,) if case["sh"] < 0 else ((case["sh"] + 1) ** 2, 3)
        values["colors"] = uniform((S, N) + colour, 0, 1)
        values["secondary_colors"] = uniform((S, N) + colour, 0, 1)
        weights = uniform((S, N, 4), 0, 1)
        values["frequency_weights"] = weights / weights.sum(-1, keepdim=True)
        values["frequency_magnitudes"] = uniform((S, N, 4), 0, 8)
        values["phases"] = uniform((S, N, 4), 0, 2 * math.pi)
    # Cameras: the first looks along +z; the others turn about the box's
    # centre by up to 25 degrees ("ring") or 8.
    middle = (near + far) / 2
    yaw = uniform((S, C), -1, 1) * math.radians(25 if case["box"] == "ring" else 8)
    if case["box"] != "ring":
        yaw[:, 0] = 0
    views = torch.zeros((S, C, 4, 4), device=device)
    views[..., 0, 0] = views[..., 2, 2] = torch.cos(yaw)
    views[..., 0, 2] = -torch.sin(yaw)
    views[..., 2, 0] = torch.sin(yaw)
    views[..., 1, 1] = views[..., 3, 3] = 1.0
    views[..., 0, 3] = middle * torch.sin(yaw)
    views[..., 2, 3] = middle * (1 - torch.cos(yaw))
    K = torch.zeros((S, C, 3, 3), device=device)
    K[..., 0, 0] = K[..., 1, 1] = case["focal"] * W
    K[..., 0, 2], K[..., 1, 2], K[..., 2, 2] = (W - 1) / 2, (H - 1) / 2, 1.0
    values["view_matrices"], values["intrinsics"] = views, K
    if case["backgrounds"]:
        values["backgrounds"] = uniform((S, C, 3), 0, 1)
    values = {k: v.float().contiguous() for k, v in values.items()}
    # Gradient images: one sign per map and image with noise over the pixels,
    # scaled like a mean over the image.
    gradients = []
    if case["train"]:
        count = S * C * W * H
        for k in {"rgb": (3,), "depth": (3, 1, 1), "all": (3, 1, 1, 3, 1)}[case["maps"]]:
            sign = torch.where(uniform((S, C, 1, 1, k), 0, 1) < 0.5, -1.0, 1.0)
            gradients.append((sign * uniform((S, C, H, W, k), 0, 2) / count).contiguous())
    return values, gradients


def _trained(case):
    return (PARAMETERS + (NEURAL if case["neural"] else CLASSIC)
            + (CAMERAS[:2] if case["poses"] else ())
            + (CAMERAS[2:] if case["backgrounds"] else ()))


def prepare(case, seed):
    values, gradients = _inputs(case, seed, torch.device("cuda"))
    if case["train"]:
        for name in _trained(case):
            values[name].requires_grad_()
    options = dict(width=case["width"], height=case["height"], packed=case["packed"],
                   validate=case["validate"])
    if not case["neural"]:
        options["sh_degree"] = None if case["sh"] < 0 else case["sh"]
    return {
        "renderer": rasterize_neural_gabors if case["neural"] else rasterize_gabors,
        "values": values,
        "options": options,
        "parameters": [values[name] for name in _trained(case)] if case["train"] else [],
        "gradients": gradients,
        "scope": (fixed_capacity(case["capacity"]) if case["capacity"]
                  else contextlib.nullcontext()),
    }


def run(state):
    """Returns the five maps, the dense radii and, in training, every gradient."""
    training = bool(state["gradients"])
    with state["scope"], torch.set_grad_enabled(training):
        rgb, alpha, meta = state["renderer"](**state["values"], **state["options"])
        maps = [rgb, alpha, meta["accumulated_depth"], meta["normals"], meta["distortion"]]
        outputs = [m.detach() for m in maps]
        if not state["options"]["packed"]:  # packed rows: as many as are visible
            outputs.append(meta["radii"])
        if training:
            used = maps[:len(state["gradients"])]
            outputs += torch.autograd.grad(used, state["parameters"], state["gradients"])
    return outputs


def _widths(case):
    colour = 3 if case["sh"] < 0 else 3 * (case["sh"] + 1) ** 2
    return 10 + (57 if case["neural"] else 2 * colour + 12)


def work(case):
    """Bytes: every parameter read once (and its gradient written once), the
    maps written once (and their gradients read once), the radii written.
    Operations: those of the samples that the image is made of, i.e. the
    records that cover a pixel with alpha >= 1/255 until it is opaque."""
    pairs = case["scenes"] * case["cameras"] * case["n"]
    pixels = case["scenes"] * case["cameras"] * case["width"] * case["height"]
    data = 4 * case["scenes"] * case["n"] * _widths(case) + 4 * pairs
    maps = 4 * MAP_CHANNELS * pixels
    half, near, far = BOXES[case["box"]]
    focal = case["focal"] * case["width"]
    # Mean footprint in pixels: pi s_u s_v rho_max f^2 / z^2 cos(tilt), with the
    # means of the scales, of 1/z^2 and of 2 ln(255 o), o in U(0.1, 0.9).
    log_ratio = math.log(case["scale_high"] / case["scale_low"])
    scale = (case["scale_high"] - case["scale_low"]) / log_ratio
    area = (math.pi * scale * scale * 9.2 * focal * focal / (near * far)
            * (1 + case["tilt"]) / 2)
    seen = min(1.0, near * far * case["width"] * case["height"] / (2 * half * focal) ** 2)
    layers = pairs * seen * area / pixels
    layers = min(layers, 60.0)  # by then a pixel is opaque
    flops = pixels * layers * ((300 if case["neural"] else 110) if not case["train"]
                               else (1000 if case["neural"] else 380))
    flops += pairs * (600 if case["train"] else 200)
    train = 2 if case["train"] else 1
    return {"bytes": train * (data + maps), "flops": flops}


def tolerance(case):
    """About four times what 32-bit results of random scenes were measured to
    be off from exact(). The distortion map decides: it is the small rest of
    a cancellation, T m^2 + m2 - 2 m m1, which is the smaller the thinner the
    visible layer is against its depth (measured: 1.4e-3 room, 2.7e-3
    clusters, 5e-3 near, 1e-2 ring; the other maps 1e-4, the gradients 2e-3
    where a sample on a threshold falls on the other side). Radii are
    ceilings: up to 9e-4 of them land on the next whole number."""
    return {"rel": {"room": 5e-3, "clusters": 1e-2, "near": 2e-2, "ring": 4e-2}[case["box"]],
            "differ": 4e-3}


# The same pass in 64 bits, plain torch ---------------------------------------

_SH = (0.28209479177387814, 0.4886025119029199, 1.0925484305920792, 0.31539156525252005,
       0.5462742152960396, 0.5900435899266435, 2.890611442640554, 0.4570457994644658,
       0.3731763325901154, 1.445305721320277)
_TILE = 16


def _sh_basis(d, degree):
    x, y, z = d.unbind(-1)
    b = [torch.full_like(x, _SH[0])]
    if degree > 0:
        b += [-_SH[1] * y, _SH[1] * z, -_SH[1] * x]
    if degree > 1:
        b += [_SH[2] * x * y, -_SH[2] * y * z, _SH[3] * (3 * z * z - 1), -_SH[2] * x * z,
              _SH[4] * (x * x - y * y)]
    if degree > 2:
        b += [-_SH[5] * y * (3 * x * x - y * y), _SH[6] * x * y * z,
              -_SH[7] * y * (5 * z * z - 1), _SH[8] * z * (5 * z * z - 3),
              -_SH[7] * x * (5 * z * z - 1), _SH[9] * z * (x * x - y * y),
              -_SH[5] * x * (x * x - 3 * y * y)]
    return torch.stack(b, -1)


def _project(p, case, scene, camera, near, far):
    """One image's records (geometry, appearance, opacity: differentiable),
    radii and tile rectangles, all [N, ...]."""
    q = p["quaternions"][scene]
    q = q / q.norm(dim=-1, keepdim=True)
    w, x, y, z = q.unbind(-1)
    axes = [torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y + w * z), 2 * (x * z - w * y)], -1),
            torch.stack([2 * (x * y - w * z), 1 - 2 * (x * x + z * z), 2 * (y * z + w * x)], -1),
            torch.stack([2 * (x * z + w * y), 2 * (y * z - w * x), 1 - 2 * (x * x + y * y)], -1)]
    view, K = p["view_matrices"][scene, camera], p["intrinsics"][scene, camera]
    R, t = view[:3, :3], view[:3, 3]
    mean, scale = p["means"][scene], p["scales"][scene]
    columns = [scale[:, :1] * axes[0] @ R.T, scale[:, 1:] * axes[1] @ R.T, mean @ R.T + t]
    T = torch.stack([c @ K.T for c in columns], -1)  # [N, 3, 3]
    f = T.new_tensor([9.0, 9.0, -1.0])
    f = f / (f * T[:, 2] ** 2).sum(-1, keepdim=True)
    xy = (f[:, None] * T[:, :2] * T[:, 2:]).sum(-1)
    extent = xy ** 2 - (f[:, None] * T[:, :2] ** 2).sum(-1)
    normal = axes[2] @ R.T
    facing = -(columns[2] * normal).sum(-1)
    normal = torch.where(facing > 0, 1.0, -1.0)[:, None] * normal
    direction = mean + R.T @ t
    direction = direction / direction.norm(dim=-1, keepdim=True)
    with torch.no_grad():
        radius = extent.clamp_min(1e-4).sqrt().amax(-1).clamp_min(3 * 0.707106).ceil()
        grid = T.new_tensor([(case["width"] + 15) // _TILE, (case["height"] + 15) // _TILE])
        low = torch.minimum(((xy - radius[:, None]) / _TILE).trunc().clamp_min(0), grid)
        high = torch.minimum(((xy + radius[:, None] + 15) / _TILE).trunc().clamp_min(0), grid)
        depth = columns[2][:, 2]
        ok = (depth > near) & (depth < far) & (facing != 0) & (radius < 2 ** 30)
        ok &= torch.isfinite(xy).all(-1) & (high > low).all(-1)
        radius = torch.where(ok, radius, torch.zeros_like(radius)).int()
    if case["neural"]:
        rows = torch.cat([p[k][scene].flatten(1) for k in NEURAL], -1)
    else:
        colours = [p[k][scene] for k in CLASSIC[:2]]
        if case["sh"] >= 0:
            basis = _sh_basis(direction, case["sh"])[..., None]
            colours = [(0.5 + (basis * c).sum(1)).clamp_min(0) for c in colours]
        rows = torch.cat(colours + [p[k][scene] for k in CLASSIC[2:]], -1)
    geometry = torch.cat([T.flatten(1), xy, normal, direction], -1)
    return torch.cat([geometry, p["opacities"][scene][:, None], rows], -1), radius, low, high


def _sample(r, x, y, neural, near):
    """Alpha (zero where a sample is not accepted), local coordinates and depth
    of records r [B, K, F] at pixels x, y [B, P]: [B, P, K]."""
    g = [r[:, None, :, i] for i in range(11)]
    o = r[:, None, :, 17]
    x, y = x[..., None], y[..., None]
    k = [x * g[6 + i] - g[i] for i in range(3)]
    l = [y * g[6 + i] - g[3 + i] for i in range(3)]  # noqa: E741
    pz = k[0] * l[1] - k[1] * l[0]
    flat = pz == 0
    pz = torch.where(flat, torch.ones_like(pz), pz)
    u = (k[1] * l[2] - k[2] * l[1]) / pz
    v = (k[2] * l[0] - k[0] * l[2]) / pz
    rho3 = u * u + v * v
    rho2 = 2 * ((g[9] - x) ** 2 + (g[10] - y) ** 2)
    depth = u * g[6] + v * g[7] + g[8]
    if not neural:
        depth = torch.where(rho3 <= rho2, depth, g[8].expand_as(depth))
    alpha = (o * torch.exp(-0.5 * torch.minimum(rho3, rho2))).clamp_max(0.99)
    ok = ~flat & (depth >= near) & (alpha >= 1.0 / 255.0)
    return alpha, u, v, depth, ok


def _taken(alpha, ok):
    """Accepted records up to the one that would take T below 1e-4."""
    return ok & (torch.cumprod(torch.where(ok, 1 - alpha, torch.ones_like(alpha)), -1) >= 1e-4)


def _shade(r, u, v, neural):
    a = r[:, None, :, 18:]
    if neural:
        d = [r[:, None, :, 14 + i] for i in range(3)]
        hidden = []
        for h in range(6):
            w = [a[..., 5 * h + i] for i in range(5)]
            z = w[0] * (u / 3) + w[1] * (v / 3) + (w[2] * d[0] + w[3] * d[1] + w[4] * d[2]
                                                   + a[..., 30 + h])
            hidden.append(torch.sin(30 * z))
        return [torch.sigmoid(sum(a[..., 36 + 6 * c + h] * hidden[h] for h in range(6))
                              + a[..., 54 + c]) for c in range(3)]
    mix = 0
    for f in range(4):
        angle = math.pi * f / 4
        dot = u * math.cos(angle) + v * math.sin(angle)
        mix = mix + a[..., 6 + f] / 2 * torch.cos(2 * math.pi * a[..., 10 + f] * dot
                                                  + a[..., 14 + f])
    half = a[..., 6:10].sum(-1) / 2
    return [(half + mix) * a[..., c] + (half - mix) * a[..., 3 + c] for c in range(3)]


def _composite(r, keep, x, y, background, neural, near, far):
    """The nine maps [B, P, 9] of tiles with records r [B, K, F]."""
    alpha, u, v, depth, _ = _sample(r, x, y, neural, near)
    zero, one = torch.zeros_like(alpha), torch.ones_like(alpha)
    alpha = torch.where(keep, alpha, zero)
    u, v = torch.where(keep, u, zero), torch.where(keep, v, zero)
    depth = torch.where(keep, depth, one)
    through = torch.cumprod(1 - alpha, -1)
    final = through[..., -1]
    T = torch.cat([one[..., :1], through[..., :-1]], -1)
    w = T * alpha
    m = far / (far - near) * (1 - near / depth)
    s1, s2 = w * m, w * m * m
    distortion = (w * (m * m * (1 - T) + torch.cumsum(s2, -1) - s2
                       - 2 * m * (torch.cumsum(s1, -1) - s1))).sum(-1)
    colour = _shade(r, u, v, neural)
    maps = [(w * colour[c]).sum(-1) + final * background[c] for c in range(3)]
    maps += [1 - final, (w * depth).sum(-1)]
    maps += [(w * r[:, None, :, 11 + i]).sum(-1) for i in range(3)]
    return torch.stack(maps + [distortion], -1)


def _image(p, case, scene, camera, gradient, background, near=0.2, far=100.0):
    """One image's maps [H, W, 9] and radii [N]; with gradient images, the
    gradients of the parameters are added to the leaves of `p`."""
    W, H, neural = case["width"], case["height"], case["neural"]
    rows, radius, low, high = _project(p, case, scene, camera, near, far)
    device = rows.device
    tw, th = (W + 15) // _TILE, (H + 15) // _TILE
    # Point lists: visible surfels by depth, expanded over their tiles.
    seen = torch.nonzero(radius > 0).squeeze(-1)
    seen = seen[torch.sort(rows.detach()[seen, 8].float(), stable=True).indices]
    x0, y0 = low[seen].long().unbind(-1)
    nx, ny = (high - low)[seen].long().unbind(-1)
    count = nx * ny
    surfel = torch.repeat_interleave(seen, count)
    start = torch.repeat_interleave(torch.cumsum(count, 0) - count, count)
    index = torch.arange(len(surfel), device=device) - start
    wide = torch.repeat_interleave(nx, count)
    tile = ((torch.repeat_interleave(y0, count) + index // wide) * tw
            + torch.repeat_interleave(x0, count) + index % wide)
    order = torch.sort(tile, stable=True)
    surfel = surfel[order.indices]
    lengths = torch.bincount(tile, minlength=tw * th)
    first = torch.cumsum(lengths, 0) - lengths
    by_length = torch.sort(lengths, descending=True).indices
    sizes = lengths[by_length].tolist()
    table = torch.cat([rows, torch.zeros_like(rows[:1])])  # the last row: no record
    leaf = table.detach().requires_grad_(gradient is not None)
    out = torch.zeros((H, W, 9), dtype=torch.float64, device=device)
    bg = background.detach().requires_grad_(gradient is not None)
    offsets = torch.arange(_TILE * _TILE, device=device)
    at = 0
    while at < tw * th:
        K = max(sizes[at], 1)
        tiles = by_length[at:at + max(1, (1 << 21) // (K * _TILE * _TILE))]
        at += len(tiles)
        slot = torch.arange(K, device=device)
        has = slot < lengths[tiles][:, None]
        where = (first[tiles][:, None] + slot).clamp_max(max(len(surfel) - 1, 0))
        ids = torch.where(has, surfel[where], len(rows)) if len(surfel) else (
            torch.full((len(tiles), K), len(rows), device=device))
        px = (tiles % tw)[:, None] * _TILE + offsets % _TILE
        py = (tiles // tw)[:, None] * _TILE + offsets // _TILE
        inside = (px < W) & (py < H)
        with torch.no_grad():
            alpha, *_, ok = _sample(leaf.detach()[ids], px.double(), py.double(), neural, near)
            keep = _taken(alpha, ok & has[:, None]) & inside[..., None]
            # Only the records that some pixel of the tile takes.
            used = keep.any(1)
            most = max(int(used.sum(1).max()), 1)
            pick = torch.sort((~used).byte(), dim=1, stable=True).indices[:, :most]
            keep = torch.gather(keep, 2, pick[:, None].expand(-1, _TILE * _TILE, -1))
            ids = torch.gather(ids, 1, pick)
        maps = _composite(leaf[ids], keep, px.double(), py.double(), bg, neural, near, far)
        py, px = py[inside], px[inside]
        out[py, px] = maps[inside].detach()
        if gradient is not None:
            (maps[inside] * gradient[py, px]).sum().backward()
    if gradient is not None:
        rows.backward(leaf.grad[:-1])
        if background.requires_grad:
            background.backward(bg.grad)
    return out, radius


def exact(case, seed):
    """What run() returns, computed densely per tile in 64 bits; None for the
    largest batch, whose 10^10 samples take too long this way."""
    if work(case)["flops"] > 0.5 * LIMIT or case["n"] * case["scenes"] * case["cameras"] > 1.1e6:
        return None
    device = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    values, gradients = _inputs(case, seed, device)
    p = {k: v.double() for k, v in values.items()}
    trained = _trained(case) if case["train"] else ()
    for name in trained:
        p[name].requires_grad_()
    S, C, H, W = case["scenes"], case["cameras"], case["height"], case["width"]
    maps = torch.zeros((S, C, H, W, 9), dtype=torch.float64, device=device)
    radii = torch.zeros((S, C, case["n"]), dtype=torch.int32, device=device)
    image_gradient = None
    if case["train"]:
        image_gradient = torch.zeros_like(maps)
        at = 0
        for g in gradients:
            image_gradient[..., at:at + g.shape[-1]] = g
            at += g.shape[-1]
    with torch.set_grad_enabled(case["train"]):
        for scene in range(S):
            for camera in range(C):
                background = (p["backgrounds"][scene, camera] if case["backgrounds"]
                              else maps.new_zeros(3))
                maps[scene, camera], radii[scene, camera] = _image(
                    p, case, scene, camera,
                    None if image_gradient is None else image_gradient[scene, camera], background)
    maps, radii = maps.cpu(), radii.reshape(-1).cpu()
    outputs = [maps[..., 0:3], maps[..., 3:4], maps[..., 4:5], maps[..., 5:8], maps[..., 8:9]]
    if not case["packed"]:
        outputs.append(radii.reshape(S, C, -1))
    outputs += [torch.zeros_like(p[k]).cpu() if p[k].grad is None else p[k].grad.cpu()
                for k in trained]
    return [t.contiguous().numpy() for t in outputs]
