"""The classic replay backward, whose lanes are 16 records x 4 pixels.

Its chunks of 16 records, its queue of filtered entries (refilled 64 at a
time) and its three variants by the gradient groups present are checked on
stacks of surfels that every pixel takes, at lengths around those sizes,
against the full-list walk, which keeps one pixel per lane, sums across the
wave and derives every row of T per pixel.

Both take the same records with the same per-sample float32 values; they
differ in the order of the sums over at most 256 pixels and n records, so a
gradient's error against the other is a few 2^-24 sqrt(256 n) of the summed
magnitudes: 1e-5 of the tensor's norm for n <= 145, with a cancellation of
up to 2 bits between the terms of one record. The distortion
goes with rgb: its own dL/dw, m^2 A + m2 - 2 m m1, keeps (dm / m)^2 ~ 6e-4 of
its terms and dL/dalpha is a difference of such values, so alone it is known
to 1e-4 at best on either side.
"""

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


def gradients(values, gradient_groups, non_finite=False):
    """(by record, full list) gradients of one render."""
    from diff_gabor_splatting_amd import _native

    args = compositor_inputs(renderer(False), values, dict(width=WIDTH, height=HEIGHT))
    maps, points, ranges, state, contributors, replay = _native.rasterize_forward(
        *args, replay=True)
    saved = (*args[:4], args[6], points, ranges, state, contributors)
    g = torch.Generator().manual_seed(7)
    groups = [torch.randn(1, HEIGHT, WIDTH, k, generator=g).to(DEVICE) if on else None
              for k, on in zip((3, 1, 1, 3, 1), gradient_groups)]
    if non_finite:
        groups[0][0, 2, 3, 1] = float("inf")
    return [_native.rasterize_backward(*saved, groups, WIDTH, HEIGHT, False, *args[10:12],
                                       replay=lists) for lists in (replay, None)]


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 79, 80, 81, 145])
@pytest.mark.parametrize("present", ["rgb", "rgb+alpha", "depth", "normals", "rgb+distortion",
                                     "all"])
def test_chunks_match_the_full_walk(n, present):
    on = {"rgb": (1, 0, 0, 0, 0), "rgb+alpha": (1, 1, 0, 0, 0), "depth": (1, 1, 1, 0, 0),
          "normals": (0, 0, 0, 1, 0), "rgb+distortion": (1, 0, 0, 0, 1), "all": (1, 1, 1, 1, 1)}
    for a, e in zip(*gradients(stack(n, n), on[present])):
        assert float((a - e).norm()) <= 1e-5 * float(e.norm())


def test_a_non_finite_pixel_reaches_only_the_records_it_took():
    values = stack(40, 3)
    values["scales"].mul_(0.2)  # most surfels miss the pixel
    for a, e in zip(*gradients(values, (1, 1, 1, 1, 1), non_finite=True)):
        assert torch.equal(torch.isfinite(a), torch.isfinite(e))
        fine = torch.isfinite(e)
        assert fine.any()
        assert float((a - e)[fine].norm()) <= 1e-5 * float(e[fine].norm())
