"""GPU checks that the sampler's single walk and its two passes (count, segments) give the same segments bit for bit,
whatever the root's box (in trees whose boxes FP32 cannot halve exactly a box depends on the way the walk took), and on
both sides of the batch size up to which a wave walks a ray."""
import numpy as np
import pytest
import torch

from neat_amd import ops, workloads as W

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rays(n, lo, hi, seed):
    g = np.random.default_rng(seed)
    size = hi - lo
    o = lo + size * g.uniform(-1, 2, (n, 3))
    d = lo + size * g.uniform(0, 1, (n, 3)) - o
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    k = n // 4  # along one axis, on the nominal faces between cells
    axis = g.integers(0, 3, k)
    o[:k] = lo + size * g.integers(0, 17, (k, 3)) / 16.0
    o[np.arange(k), axis] = (lo - size)[axis]
    d[:k] = 0
    d[np.arange(k), axis] = 1
    return torch.from_numpy(o.astype(np.float32)).to(DEV), torch.from_numpy(d.astype(np.float32)).to(DEV)


def check(n, depth, lo, hi, kind="leaves"):
    t = W.build_tree(depth)
    act = (t["depth"] == depth).astype(np.int32)
    if kind == "overlap":
        act = (np.random.default_rng(2).random(t["depth"].shape[0]) < 0.2).astype(np.int32)
        act[0] = 1
    lo, hi = np.asarray(lo, np.float64), np.asarray(hi, np.float64)
    pmin, pmax = (torch.from_numpy((lo + (t[k] + 1) / 2 * (hi - lo)).astype(np.float32)).to(DEV)
                  for k in ("pos_min", "pos_max"))
    flags = ops.tree_flags(act, depth).to(DEV)
    o, d = rays(n, lo, hi, depth + n)
    a = ops.raysample(pmin, pmax, flags, depth, o, d, 16, emit=False)
    b = ops.raysample(pmin, pmax, flags, depth, o, d, 16, emit=False, single_walk=False)
    assert b["seg_node"].shape[0] > 0 or n == 1
    for k, v in b.items():
        if torch.is_tensor(v):
            assert torch.equal(a[k], v), k
        else:
            assert a[k] == v, k


@pytest.mark.parametrize("box", [((0, 0, 0), (3, 3, 3)), ((-0.7, -0.7, -0.7), (1.3, 1.3, 1.3)),
                                 ((-1, -1, 0.1), (1, 1, 0.7)), ((-8388607, -1, -1), (8388607, 1, 1)),
                                 ((-0.83, -1.7, -2.9), (0.83, 1.7, 2.9))])
@pytest.mark.parametrize("depth,kind,n", [(0, "leaves", 3), (2, "leaves", 701), (5, "overlap", 700), (5, "leaves", 5001),
                                          (6, "leaves", 301)])
def test_root_box(depth, kind, n, box):
    print("case: sampler, root box", depth, kind, n, box, flush=True)
    check(n, depth, *box, kind)


@pytest.mark.parametrize("depth,n", [(2, 2047), (2, 2048), (2, 2049), (3, 6144), (3, 6145), (5, 65535), (5, 65536),
                                     (5, 65537)])
def test_batch_limits(depth, n):
    print("case: sampler, batch limits", depth, n, flush=True)
    check(n, depth, (-1, -1, -1), (1, 1, 1))
