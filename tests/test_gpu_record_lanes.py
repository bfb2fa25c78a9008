"""The classic replay backward, whose lanes are 16 records x 4 pixels.

Its chunks of 16 records, its windows of 128 or 192 entries and its three
variants by the gradient groups present are checked on stacks of surfels that
every pixel takes, at lengths around those sizes, against the full-list walk,
which keeps one pixel per lane, sums across the wave and derives every row of T
per pixel.

Both take the same records with the same per-sample float32 values; they
differ in the order of the sums over at most 256 pixels and n records, so a
gradient's error against the other is a few 2^-24 sqrt(256 n) of the summed
magnitudes: 1e-5 of the tensor's norm for n <= 145, with a cancellation of
up to 2 bits between the terms of one record. The distortion
goes with rgb: its own dL/dw, m^2 A + m2 - 2 m m1, keeps (dm / m)^2 ~ 6e-4 of
its terms and dL/dalpha is a difference of such values, so alone it is known
to 1e-4 at best on either side.
"""

import math

import pytest
import torch

from test_gpu_replay import compositor_inputs, renderer

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]
DEVICE = torch.device("cuda:0")
WIDTH, HEIGHT = 21, 19  # two ragged tiles each way


def stack(n, seed):
    """n translucent surfels in front of a small camera, tilted by up to 60
    degrees, with about half covering every pixel."""
    g = torch.Generator().manual_seed(seed)

    def uniform(shape, low, high):
        return torch.rand(shape, generator=g) * (high - low) + low

    angle, axis = uniform((1, n), -0.5, 0.5), uniform((1, n), 0, 6.28)
    weights = uniform((1, n, 4), 0, 1)
    values = dict(
        means=torch.cat([uniform((1, n, 2), -0.3, 0.3), uniform((1, n, 1), 2, 4)], -1),
        quaternions=torch.stack([angle.cos(), angle.sin() * axis.cos(), angle.sin() * axis.sin(),
                                 torch.zeros(1, n)], -1),
        scales=uniform((1, n, 2), 0.1, 0.9), opacities=uniform((1, n), 0.02, 0.06),
        colors=uniform((1, n, 3), 0, 1), secondary_colors=uniform((1, n, 3), 0, 1),
        frequency_weights=weights / weights.sum(-1, keepdim=True),
        frequency_magnitudes=uniform((1, n, 4), 0, 3), phases=uniform((1, n, 4), 0, 6.28),
        view_matrices=torch.eye(4)[None, None],
        intrinsics=torch.tensor([[[[20.0, 0, 10], [0, 20.0, 9], [0, 0, 1.0]]]]),
        backgrounds=uniform((1, 1, 3), 0, 1))
    return {k: v.contiguous().to(DEVICE) for k, v in values.items()}


GROUPS = {"rgb": (1, 0, 0, 0, 0), "rgb+alpha": (1, 1, 0, 0, 0), "depth": (1, 1, 1, 0, 0),
          "normals": (0, 0, 0, 1, 0), "rgb+distortion": (1, 0, 0, 0, 1), "all": (1, 1, 1, 1, 1)}


def gradients(values, gradient_groups, non_finite=False, width=WIDTH, height=HEIGHT):
    """(by record, full list) gradients of one render."""
    from diff_gabor_splatting_amd import _native

    args = compositor_inputs(renderer(False), values, dict(width=width, height=height))
    maps, points, ranges, state, contributors, replay = _native.rasterize_forward(
        *args, replay=True)
    saved = (*args[:4], args[6], points, ranges, state, contributors)
    g = torch.Generator().manual_seed(7)
    groups = [torch.randn(1, height, width, k, generator=g).to(DEVICE) if on else None
              for k, on in zip((3, 1, 1, 3, 1), gradient_groups)]
    if non_finite:
        groups[0][0, 2, 3, 1] = float("inf")
    return [_native.rasterize_backward(*saved, groups, width, height, False, *args[10:12],
                                       replay=lists) for lists in (replay, None)]


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 79, 80, 81, 145])
@pytest.mark.parametrize("present", ["rgb", "rgb+alpha", "depth", "normals", "rgb+distortion",
                                     "all"])
def test_chunks_match_the_full_walk(n, present):
    for a, e in zip(*gradients(stack(n, n), GROUPS[present])):
        assert float((a - e).norm()) <= 1e-5 * float(e.norm())


@pytest.mark.parametrize("n", [2, 3, 4, 5, 7, 8, 9, 11, 12, 13, 28, 29])
@pytest.mark.parametrize("present", ["rgb", "depth", "all"])
def test_few_records_match_the_full_walk(n, present):
    """Up to 12 records, and as many left after a chunk of 16, go in chunks of
    four; a chunk's last one may be partly filled."""
    values = stack(n, n)
    values["scales"].mul_(2)  # most cover every pixel, so that all quadrants hold n
    for a, e in zip(*gradients(values, GROUPS[present])):
        assert float((a - e).norm()) <= 1e-5 * float(e.norm())


@pytest.mark.parametrize("scene", ["few records per tile", "surfels that fill the image"])
def test_not_slower_than_a_pixel_per_lane(scene):
    """The full-list walk evaluates a pixel per lane. Where tiles hold few records
    (a chunk's cost whatever it holds) or a record spans all of them (its atomics
    follow each other) the walk by record must not lose to it. Measured 0.94 and
    0.72 of its time; with chunks of 16 only, the first 1.4; with an atomic per
    quadrant, the second 2.4."""
    from diff_gabor_splatting_amd import _native

    width, height = 1920, 1080
    few = scene.startswith("few")
    values = stack(10_000 if few else 16, 2)
    g = torch.Generator().manual_seed(8)
    n = values["means"].shape[1]
    spread = torch.tensor([2.5, 1.5]) * (torch.rand(1, n, 2, generator=g) * 2 - 1)
    if few:
        values["means"][..., :2] = spread.to(DEVICE)
        values["scales"].mul_(0.03)
    else:
        values["scales"].fill_(5.0)
    values["intrinsics"] = torch.tensor(
        [[[[1900.0, 0, 960], [0, 1900.0, 540], [0, 0, 1.0]]]], device=DEVICE)
    args = compositor_inputs(renderer(False), values, dict(width=width, height=height))
    _, points, ranges, state, contributors, replay = _native.rasterize_forward(*args, replay=True)
    saved = (*args[:4], args[6], points, ranges, state, contributors)
    groups = [torch.randn(1, height, width, k, device=DEVICE) for k in (3, 1, 1, 3, 1)]
    accumulators = _native.zero_accumulators(args[0], args[1], args[2], args[6])

    def median(lists):
        times = []
        for _ in range(25):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            _native.rasterize_backward(*saved, groups, width, height, False, *args[10:12],
                                       accumulators=accumulators, replay=lists)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        return sorted(times)[len(times) // 2]

    by_record, by_pixel = median(replay), median(None)
    print(f"{scene}: {1e3 * by_record:.0f} us, a pixel per lane {1e3 * by_pixel:.0f}", flush=True)
    assert by_record <= 1.2 * by_pixel


@pytest.mark.parametrize("n", [127, 128, 129, 191, 192, 193, 257, 400])
@pytest.mark.parametrize("present", ["rgb", "depth", "all"])
def test_windows_match_the_full_walk(n, present):
    """Lists around the windows' edges (128 entries, with all maps 192) and of
    several windows. The bound grows with the root of the list's length from
    the 1e-5 at 145."""
    values = stack(n, n)
    values["opacities"].mul_(0.4)  # some 400 records before a pixel stops
    for a, e in zip(*gradients(values, GROUPS[present])):
        assert float((a - e).norm()) <= 1e-5 * max(1, n / 145) ** 0.5 * float(e.norm())


@pytest.mark.parametrize("present", ["rgb", "depth", "all"])
def test_centres_far_from_the_tile(present):
    """Wide and steeply tilted surfels whose centres lie more than the 64 pixels
    away that the moment sums' reference point is held within. There the sums
    about that point and the rows of T about it are both of the size of the
    affine functions k and l at the pixel (both grow with the distance), so the
    bound stays that of the other scenes."""
    n, width, height = 60, 640, 40
    values = stack(n, 5)
    g = torch.Generator().manual_seed(6)

    def uniform(low, high):
        return torch.rand(1, n, generator=g) * (high - low) + low

    values["means"][..., 0] = uniform(-2.5, 2.5).to(DEVICE)
    values["scales"][..., 0] = uniform(0.5, 4.0).to(DEVICE)
    angle = uniform(-0.7, 0.7)  # half the rotation about y: up to 80 degrees
    zero = torch.zeros_like(angle)
    values["quaternions"] = torch.stack([angle.cos(), zero, angle.sin(), zero], -1).to(DEVICE)
    values["intrinsics"] = torch.tensor(
        [[[[300.0, 0, 320], [0, 300.0, 20], [0, 0, 1.0]]]], device=DEVICE)
    args = compositor_inputs(renderer(False), values, dict(width=width, height=height))
    from diff_gabor_splatting_amd import _native

    _, points, ranges, _, _, (lists, counts, _) = _native.rasterize_forward(*args, replay=True)
    far = 0
    for tile, ((first, _), count) in enumerate(zip(ranges.tolist(), counts.tolist())):
        centre = 16 * (tile % (width // 16)) + 7.5
        x = args[0][lists[first:first + count, 0].long(), 9]
        far += int(((x - centre).abs() > 64).sum())
    print(f"{far} records of tiles with a centre more than 64 px away", flush=True)
    assert far > 200
    for a, e in zip(*gradients(values, GROUPS[present], width=width, height=height)):
        assert float((a - e).norm()) <= 1e-5 * float(e.norm())


def test_a_record_rounds_once_per_tile():
    """A record's gradient takes one atomic addition per tile, not one per
    quadrant: m additions of one sign round by ulp / sqrt(12) each, on average
    2.5e-8 of the partial sum, in all 2.5e-8 sqrt(m / 3) of the total. m = 1,024
    tiles give 4.6e-7 and 4,096 quadrants 9.2e-7; the root mean square over 48
    sums is known to a tenth of itself, and the bound lies between."""
    from diff_gabor_splatting_amd import _native

    images, size = 16, 512
    values = stack(1, 1)
    values["means"] = torch.tensor([[[0.0, 0.0, 2.0]]], device=DEVICE)
    values["quaternions"] = torch.tensor([[[1.0, 0, 0, 0]]], device=DEVICE)
    values["scales"] = torch.full((1, 1, 2), 50.0, device=DEVICE)
    values["view_matrices"] = torch.eye(4, device=DEVICE).repeat(1, images, 1, 1)
    values["intrinsics"] = torch.tensor(
        [[400.0, 0, 256], [0, 400.0, 256], [0, 0, 1.0]], device=DEVICE).repeat(1, images, 1, 1)
    values["backgrounds"] = torch.zeros(1, images, 3, device=DEVICE)
    args = list(compositor_inputs(renderer(False), values, dict(width=size, height=size)))
    args[2] = torch.full_like(args[2], 4.0)  # alpha = 0.99 at every pixel
    _, points, ranges, state, contributors, replay = _native.rasterize_forward(*args, replay=True)
    assert bool((contributors == 1).all())
    g = torch.Generator(device=DEVICE).manual_seed(3)
    normals = torch.rand(images, size, size, 3, generator=g, device=DEVICE) + 0.5
    saved = (*args[:4], args[6], points, ranges, state, contributors)
    geometry = _native.rasterize_backward(*saved, [None, None, None, normals, None], size, size,
                                          False, *args[10:12], replay=replay)[0]
    expected = float(torch.tensor(0.99)) * normals.double().sum((1, 2))
    error = (geometry[:, 11:14].double() - expected) / expected
    rms = float(error.square().mean().sqrt())
    print(f"relative error {rms:.2e}", flush=True)
    assert math.isfinite(rms) and rms <= 6.6e-7


def test_a_non_finite_pixel_reaches_only_the_records_it_took():
    values = stack(40, 3)
    values["scales"].mul_(0.2)  # most surfels miss the pixel
    for a, e in zip(*gradients(values, (1, 1, 1, 1, 1), non_finite=True)):
        assert torch.equal(torch.isfinite(a), torch.isfinite(e))
        fine = torch.isfinite(e)
        assert fine.any()
        assert float((a - e)[fine].norm()) <= 1e-5 * float(e[fine].norm())


def test_transmittance_does_not_drift():
    """The transmittance that the backward walks back from the last record is a
    product of n reciprocals; a reciprocal that errs to one side adds up. Surfels
    so wide that alpha is the opacity at every pixel give the weights in closed
    form, and the mean error over 64 lists leaves the one-sided part: n = 120
    records round 2 n times by 2.5e-8, 3.9e-7 a list and 5e-8 in the mean, and
    sums of 256 equal values by up to 1e-7; the bound is three and one of these."""
    from diff_gabor_splatting_amd import _native

    scenes, n, size = 64, 120, 16
    values = {k: v.expand(scenes, *v.shape[1:]).contiguous() for k, v in stack(n, 4).items()}
    g = torch.Generator().manual_seed(4)
    values["opacities"] = (torch.rand(scenes, n, generator=g) * 0.006 + 0.004).to(DEVICE)
    values["means"] = torch.cat([torch.zeros(n, 2), torch.linspace(2, 4, n)[:, None]], -1).expand(
        scenes, n, 3).contiguous().to(DEVICE)
    values["quaternions"] = torch.tensor([1.0, 0, 0, 0], device=DEVICE).repeat(scenes, n, 1)
    values["scales"] = torch.full((scenes, n, 2), 2e4, device=DEVICE)
    args = compositor_inputs(renderer(False), values, dict(width=size, height=size))
    _, points, ranges, state, contributors, replay = _native.rasterize_forward(
        *args, replay=True, split=0)
    assert bool((contributors == n).all())
    saved = (*args[:4], args[6], points, ranges, state, contributors)
    normals = torch.ones(scenes, size, size, 3, device=DEVICE)
    opacity = values["opacities"].double()
    keep = (1 - opacity).cumprod(1)
    weight = size * size * opacity * torch.cat([torch.ones_like(keep[:, :1]), keep[:, :-1]], 1)
    for lists in (replay, None):
        geometry = _native.rasterize_backward(*saved, [None, None, None, normals, None], size, size,
                                              False, *args[10:12], replay=lists)[0]
        error = (geometry[:, 13].double().reshape(scenes, n).abs() - weight) / weight
        front = float(error[:, :20].mean())
        print(f"mean relative error {front:.2e}", flush=True)
        assert abs(front) <= 2.5e-7
