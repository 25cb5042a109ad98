"""GPU check of the plan's stable sort of the segments by slot (counting sorts of one or two digits; the general radix
sort for more than 16 bits of key, for few segments and for many of more than 13 bits) against torch's stable sort: whole numbers, equal. Sizes at the tile's edges
(2048 segments), slot counts at the digits' (8 and 16 bits of key), nodes outside the grid and without a slot."""
import pytest
import torch

from neat_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def sorted_order(K, N, num_nodes, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    node = torch.randint(-1, num_nodes + 2, (K,), device=DEV, generator=gen, dtype=torch.int32)
    prefix = torch.randperm(num_nodes, device=DEV, generator=gen) - num_nodes // 8  # some nodes without a slot
    R = 3
    cuts = torch.tensor([0, K // 3, K // 2, K], device=DEV)
    ray = torch.bucketize(torch.arange(K, device=DEV), cuts[1:], right=True).int()
    segs = dict(ray_seg_offset=cuts, ray_sample_offset=cuts, seg_node=node, seg_ray=ray,
                seg_count=torch.ones(K, dtype=torch.int32, device=DEV),
                seg_tmin=torch.zeros(K, device=DEV), seg_tmax=torch.ones(K, device=DEV))
    box = torch.zeros(num_nodes, 3, device=DEV)
    o = torch.zeros(R, 3, device=DEV)
    grid = torch.zeros(N, 2, 2, 2, 8, device=DEV).permute(0, 4, 1, 2, 3)
    mlp = dict(hidden=32, layers=1, out=1, act="relu", last_act="softplus", beta=2.0, **{"in": 8})
    params = torch.zeros(8 * 32 + 32 + 32 * 32 + 32 + 32 + 1, device=DEV)
    pj = ops.Projector(box, box + 1, prefix, o, o + 1, segs, grid, params, mlp)
    valid = (node >= 0) & (node < num_nodes)
    slot = torch.where(valid, prefix[node.clamp(0, num_nodes - 1).long()], -1)
    key = torch.where((slot >= 0) & (slot < N), slot, N)
    return pj.ws[:4 * K].view(torch.int32).long(), key.sort(stable=True).indices


@pytest.mark.parametrize("N", [1, 200, 255, 256, 4096, 65534, 65535])
@pytest.mark.parametrize("K", [1, 63, 2047, 2048, 2049, 4096, 4097, 70001, 1000003, (1 << 21) + 1])
def test_plan_sort(K, N):
    print("case: plan sort", K, N, flush=True)
    got, want = sorted_order(K, N, N + N // 4 + 3, K + N)
    assert torch.equal(got, want)
