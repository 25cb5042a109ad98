"""GPU checks of the sampler with a wave per ray (small batches) against the count and segment walks of a thread per ray,
bit for bit, on trees and rays that reach its limits: rays along faces and edges of the tree, axis-parallel rays, rays
that start inside, overlapping active sets (an active node with active descendants), trees whose rays cross more nodes
than its lists hold."""
import numpy as np
import pytest
import torch

from neat_amd import ops, workloads as W

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rays(n, seed):
    g = np.random.default_rng(seed)
    o = g.uniform(-2.5, 2.5, (n, 3))
    d = g.uniform(-1, 1, (n, 3)) - o
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    k = n // 3
    grid = g.integers(-8, 9, (k, 3)) / 8.0  # on cell faces and edges
    axis = g.integers(0, 3, k)
    o[:k] = grid
    o[np.arange(k), axis] = g.choice([-2.0, 2.0, 0.125], k)
    d[:k] = 0
    d[np.arange(k), axis] = -np.sign(o[np.arange(k), axis])
    diag = slice(k, k + k // 4)  # through cell edges
    o[diag] = [-2, -2, 0.25]
    d[diag] = [np.sqrt(0.5), np.sqrt(0.5), 0]
    return torch.from_numpy(o.astype(np.float32)).to(DEV), torch.from_numpy(d.astype(np.float32)).to(DEV)


@pytest.mark.parametrize("n", [1, 3, 64, 701])
@pytest.mark.parametrize("depth,kind", [(0, "all"), (2, "leaves"), (4, "leaves"), (5, "adaptive"), (5, "overlap"),
                                        (6, "leaves")])
def test_wave_per_ray_matches_thread_per_ray(depth, kind, n):
    print("case: sampler, wave per ray", depth, kind, n, flush=True)
    t = W.build_tree(depth)
    if kind == "adaptive":
        act = W.adaptive_active(t, W.random_phantom(20, 3), 400, 0)
    elif kind == "overlap":
        act = (np.random.default_rng(2).random(t["depth"].shape[0]) < 0.2).astype(np.int32)
        act[0] = 1
    else:
        act = (t["depth"] == depth).astype(np.int32)
    pmin, pmax = (torch.from_numpy(t[k]).to(DEV) for k in ("pos_min", "pos_max"))
    flags = ops.tree_flags(act, depth).to(DEV)
    o, d = rays(n, depth + n)
    a = ops.raysample(pmin, pmax, flags, depth, o, d, 16, emit=False)
    b = ops.raysample(pmin, pmax, flags, depth, o, d, 16, emit=False, single_walk=False)
    for k, v in b.items():
        if torch.is_tensor(v):
            assert torch.equal(a[k], v), k
        else:
            assert a[k] == v, k


@pytest.mark.parametrize("n", [32767, 32768, 32769, 70001])
def test_offsets_over_scan_forms(n):
    """The ray offsets at the one-launch scan's limit, against torch's cumulative sums."""
    print("case: sampler offsets", n, flush=True)
    t = W.build_tree(2)
    act = (t["depth"] == 2).astype(np.int32)
    pmin, pmax = (torch.from_numpy(t[k]).to(DEV) for k in ("pos_min", "pos_max"))
    o, d = rays(n, n)
    r = ops.raysample(pmin, pmax, ops.tree_flags(act, 2).to(DEV), 2, o, d, 16, emit=False)
    ray = r["seg_ray"].long()
    nseg = torch.bincount(ray, minlength=n)
    nsmp = torch.zeros(n, dtype=torch.int64, device=DEV).index_add_(0, ray, r["seg_count"].long())
    assert torch.equal(r["ray_seg_offset"][1:], nseg.cumsum(0)) and int(r["ray_seg_offset"][0]) == 0
    assert torch.equal(r["ray_sample_offset"][1:], nsmp.cumsum(0)) and int(r["ray_sample_offset"][0]) == 0
    assert r["max_samples_per_ray"] == int(nsmp.max())


def test_totals_need_pinned_memory():
    from neat_amd import _abi
    print("case: sampler totals", flush=True)
    off = torch.tensor([0, 3, 7], dtype=torch.int64, device=DEV)
    mx = torch.tensor([4], dtype=torch.int32, device=DEV)
    out = torch.empty(3, dtype=torch.int64, pin_memory=True)
    _abi.call("neat_raysample_totals", _abi.stream_ptr(), _abi.ptr(off), _abi.ptr(off), _abi.ptr(mx), 2, _abi.ptr(out))
    assert out.tolist() == [7, 7, 4]
    for bad in (torch.empty(3, dtype=torch.int64), torch.empty(3, dtype=torch.int64, device=DEV)):
        with pytest.raises(_abi.NeatError):
            _abi.call("neat_raysample_totals", _abi.stream_ptr(), _abi.ptr(off), _abi.ptr(off), _abi.ptr(mx), 2,
                      _abi.ptr(bad))
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert _abi.stream_ptr().value == side.cuda_stream
