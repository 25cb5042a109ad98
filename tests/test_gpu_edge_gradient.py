"""GPU check of the fused edge loss's gradient for channel counts whose atomics are gathered per wave (whole channel quads
of a channels-last grid) and for others, against the chain of steps (neighbour rows, grid sample and back)."""
import pytest
import torch

from neat_amd import ops, workloads as W

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rel(a, b):
    return float((a.double() - b).norm() / b.norm().clamp(min=1e-30))


@pytest.mark.parametrize("C", [4, 6, 12])
def test_edge_gradient_channel_counts(C):
    """The fused edge loss and its chain of steps agree for whole channel quads (the gathered atomics) and others."""
    print("case: edge gradient", C, flush=True)
    tree = W.build_tree(3)
    active = W.adaptive_active(tree, W.random_phantom(20, 3), 60, 0)
    ids, prefix = W.update_active(active)
    d = [torch.from_numpy(a).to(DEV) for a in (tree["pos_min"], tree["pos_max"])]
    flags, pre, tid = ops.tree_flags(active, 3).to(DEV), torch.from_numpy(prefix).to(DEV), torch.from_numpy(ids).to(DEV)
    grid = torch.from_numpy(W.feature_grid(len(ids) + 1, C, 5, 2, std=0.3)).to(DEV).contiguous(
        memory_format=torch.channels_last_3d)
    la, ga = ops.volume_regularizer(*d, flags, pre, tid, grid, 0.0, 1e-3, seed=9)
    lb, gb = ops.volume_regularizer_unfused(*d, flags, pre, tid, grid, 0.0, 1e-3, seed=9)
    assert abs(la.item() - lb.item()) <= 1e-6 * abs(lb.item())
    assert rel(ga, gb.double()) <= 1e-6  # a few roundings of 2^-24 per term, in another order
