"""GPU checks of the regulariser's channel-quad forms: the total variation by quads against the entry-by-entry form
(other layout, or a base address off 16 bytes), whose per-entry arithmetic is the same, so gradients are bit-equal and
losses differ by the order of FP64 sums only; the edge loss with two quads a lane against its chain of steps."""
import pytest
import torch

from neat_amd import ops, workloads as W

pytestmark = pytest.mark.gpu
DEV = "cuda"


def tv(grid, slots, overwrite, g0):
    gg = torch.empty_like(grid)
    gg.copy_(g0)
    loss = ops.tv_loss_fwd_bwd(grid, slots, 0.7, torch.full((1,), 1.5, device=DEV), gg, overwrite=overwrite)
    ga = torch.empty_like(grid)
    ga.copy_(g0)
    ops.tv_loss_bwd(grid, slots, 0.7, torch.full((1,), 1.5, device=DEV), ga)
    return loss.item(), gg, ga


@pytest.mark.parametrize("overwrite", [True, False])
@pytest.mark.parametrize("C,G", [(4, 2), (4, 17), (8, 5), (8, 17), (12, 3), (6, 5)])
def test_tv_quads(C, G, overwrite):
    print("case: tv quads", C, G, overwrite, flush=True)
    N = 5
    gen = torch.Generator(device=DEV).manual_seed(C * G)
    x = torch.randint(-2, 3, (N, C, G, G, G), device=DEV, generator=gen) / 4.0  # equal neighbours among them
    x[3, 0, 0, 0, 0] = float("inf")
    x[3, 1, 1, 1, 1] = -0.0
    g0 = torch.randn(N, C, G, G, G, device=DEV, generator=gen)
    slots = torch.tensor([3, 0, 4], device=DEV)
    cl = x.contiguous(memory_format=torch.channels_last_3d)
    raw = torch.empty(x.numel() + 1, device=DEV)[1:]  # the same layout, 4 bytes off
    off = raw.view(N, G, G, G, C).permute(0, 4, 1, 2, 3)
    off.copy_(x)
    a = tv(cl, slots, overwrite, g0)
    for b in (tv(x, slots, overwrite, g0), tv(off, slots, overwrite, g0)):
        assert a[0] == b[0] or abs(a[0] - b[0]) <= 1e-12 * abs(b[0])
        assert torch.equal(a[1], b[1]) and torch.equal(a[2], b[2])


@pytest.mark.parametrize("C", [8, 16, 20])
def test_edge_two_quads(C):
    print("case: edge two quads", C, flush=True)
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
    # a few roundings of 2^-24 per term, in another order
    assert float((ga.double() - gb.double()).norm() / gb.double().norm()) <= 1e-6
    # the loss alone sums in the same order
    lo = ops.edge_loss_direct(*d, flags, pre, tid, grid, 9, 1e-3)
    assert lo.item() == la.item()
