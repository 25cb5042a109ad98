"""GPU check (the size query asks the sort library, which asks the device) that the projector's workspace grows with the
segments, the samples and the slots, so that one sized for a program's largest batch and tree serves all smaller ones."""
import ctypes

import pytest
import torch

from neat_amd import _abi

pytestmark = pytest.mark.gpu

SEGMENTS = [0, 1, 2, 100, 2047, 4095, 4096, 4097, 6143, 20000, 400000, 1 << 20, (1 << 21) - 1, 1 << 21, (1 << 21) + 1,
            2100000, 3000000, 12000000, 100000000]
SLOTS = [1, 64, 127, 128, 254, 255, 256, 511, 4095, 4096, 8190, 8191, 8192, 30000, 65534, 65535, 65536, 70000]


def size(K, S, N):
    """neat_projector_workspace_bytes, which reads the sizes and no array."""
    a = _abi.ProjectorArgs()
    for f in ("node_pos_min", "node_pos_max", "node_active_prefix_sum", "ray_origin", "ray_direction", "ray_seg_offset",
              "seg_node", "seg_ray", "seg_count", "seg_tmin", "seg_tmax", "grid", "params"):
        setattr(a, f, 4096)
    G, C = 3, 8  # the smallest grids: their share, which grows with the slots, hides nothing
    a.num_nodes, a.num_rays, a.num_segments, a.num_samples, a.num_slots = 9, 16, K, S, N
    a.channels, a.grid_size, a.in_features, a.hidden, a.hidden_layers, a.out_features = C, G, C, 32, 1, 1
    a.act, a.last_act, a.softplus_beta = _abi.ACT["relu"], _abi.ACT["softplus"], 2.0
    for i, v in enumerate((G ** 3 * C, 1, G * G * C, G * C, C)):
        a.grid_strides[i] = v
    n = _abi.lib().neat_projector_workspace_bytes(ctypes.byref(a))
    assert n > 0, _abi.last_error()
    return n


@pytest.mark.parametrize("fixed", SLOTS)
def test_grows_with_segments(fixed):
    print("case: workspace growth, slots", fixed, flush=True)
    torch.zeros(1, device="cuda")
    sizes = [size(K, 1 << 30, fixed) for K in SEGMENTS]
    assert sizes == sorted(sizes), list(zip(SEGMENTS, sizes))


@pytest.mark.parametrize("fixed", SEGMENTS)
def test_grows_with_slots(fixed):
    print("case: workspace growth, segments", fixed, flush=True)
    torch.zeros(1, device="cuda")
    sizes = [size(fixed, 1 << 30, N) for N in SLOTS]
    assert sizes == sorted(sizes), list(zip(SLOTS, sizes))
