"""The finiteness check at the edges of its 16-byte loads and 4096-value
workgroups: every planted non-finite value is found, whatever the tensor's
length modulo 4 and whether it starts on 16 bytes, and no value next to the
tensor is read into the verdict."""

import math

import pytest
import torch

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]
DEVICE = torch.device("cuda:0")


@pytest.mark.parametrize("offset", [0, 1, 4])
@pytest.mark.parametrize("count", [1, 3, 4, 5, 1023, 4095, 4096, 4097, 8191, 8195])
def test_planted_values_are_found_at_every_edge(count, offset):
    from diff_gabor_splatting_amd import _native

    store = torch.full((count + 16,), math.nan, device=DEVICE)
    tensor = store[offset:offset + count]
    tensor.fill_(3e38)  # finite, and so is its product with zero
    none = torch.empty(0, device=DEVICE)
    cameras = (torch.empty(0, 4, 4, device=DEVICE), torch.empty(0, 3, 3, device=DEVICE))

    def word():
        return int(_native.check_values([tensor], none.view(0, 4), none.view(0, 2), none,
                                        *cameras, None, None))

    assert word() == 0
    places = {0, count // 2, count - 1, (count // 4) * 4 - 1, (count // 4) * 4, 4095, 4096}
    for place in sorted(p for p in places if 0 <= p < count):
        for value in (math.inf, -math.inf, math.nan):
            tensor[place] = value
            assert word() == 1, (place, value)
        tensor[place] = -3e38
    assert word() == 0
