"""GPU check of the channels-last grid sample with two lanes a sample (whole pairs of channel quads) and one, against the
form for any strides on the same values: the same operations per channel, so bit-equal."""
import pytest
import torch

from neat_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("C", [4, 8, 12, 16, 24])
@pytest.mark.parametrize("S", [1, 127, 128, 129, 5003])
def test_grid_sample_layouts(S, C):
    print("case: grid sample forward", S, C, flush=True)
    g = torch.Generator(device=DEV).manual_seed(S * C)
    grid = torch.randn(3, C, 3, 4, 5, device=DEV, generator=g)
    uv = torch.rand(S, 3, device=DEV, generator=g) * 2.4 - 1.2  # some outside the grid
    slot = torch.randint(-1, 4, (S,), device=DEV, generator=g)  # some without a slot
    a = ops.gs3d_fwd(grid.contiguous(memory_format=torch.channels_last_3d), slot, uv)
    assert torch.equal(a, ops.gs3d_fwd(grid, slot, uv))
