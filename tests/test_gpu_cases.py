"""The performance cases' passes, output by output, against their 64-bit results.

A case has one tolerance for all its outputs, and the distortion map, the small
rest of a cancellation, decides it (5e-3 to 4e-2 of its norm). The other maps
and the gradients are known far better: a sample on a threshold that falls on
the other side shows at 1e-4 of a map and 2e-3 of a gradient in the worst of
random scenes (their float32 rounding at 1e-6 to 1e-5), and the bounds here are
five times these.
"""

import pytest
import torch

from perf import cases

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]
MAPS = ("rgb", "alpha", "depth", "normals", "distortion")


@pytest.mark.parametrize("name", ["train_small", "train_views", "train_views_neural",
                                  "train_ragged", "render_stream"])
def test_every_output_is_close_to_64_bits(name):
    case = next(c for c in cases.listed() if c["name"] == name)
    print(f"case {name}", flush=True)
    state = cases.prepare(case, 1)
    outputs, exact = cases.run(state), cases.exact(case, 1)
    assert len(outputs) == len(exact) > len(MAPS)
    gradients = len(MAPS) + (not case["packed"])  # the radii are not packed
    for i, (a, e) in enumerate(zip(outputs, exact)):
        if e is None:
            continue
        a, e = a.double().cpu(), torch.as_tensor(e).double().cpu()
        if i == len(MAPS) and not case["packed"]:
            assert float((a != e).double().mean()) <= cases.tolerance(case)["differ"]
            continue
        bound = 5e-4 if i < 4 else cases.tolerance(case)["rel"] if i == 4 else 1e-2
        error = float((a - e).norm() / e.norm())
        print(f"{MAPS[i] if i < len(MAPS) else f'gradient {i - gradients}'} {error:.1e}", flush=True)
        assert error <= bound
