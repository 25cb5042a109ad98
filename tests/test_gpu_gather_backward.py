"""GPU checks of the grid sample's backward on channels-last gradients (neat_gs3d_bwd's run-merging kernel) against the
same sums in float64 at the kernel's own FP32 grid coordinates: gradients within 1e-6 (norm-wise; every term carries
a handful of roundings of 2^-24 and a vertex adds fewer than a thousand of them), invalid slots included."""
import numpy as np
import pytest
import torch

from neat_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def reference(grid, index, uv, gout):
    """float64 (grad_grid, grad_uv) of the trilinear sample, the coordinates rounded as FP32 does."""
    N, C, Z, Y, X = grid.shape
    size = torch.tensor([X, Y, Z], device=uv.device)
    x = ((uv + 1) / 2) * (size - 1).float()
    x0 = torch.floor(x)
    f = (x - x0).double()
    i0 = x0.long()
    ok = (index >= 0) & (index < N)
    n = torch.where(ok, index, 0)
    flat = grid.permute(0, 2, 3, 4, 1).reshape(-1, C).double()
    go = torch.where(ok[:, None], gout.double(), 0.0)
    gg = torch.zeros_like(flat)
    guv = torch.zeros(len(index), 3, dtype=torch.float64, device=uv.device)
    for k in range(8):
        b = [(k >> a) & 1 for a in range(3)]
        c = [torch.minimum((i0[:, a] + b[a]).clamp(min=0), size[a] - 1) for a in range(3)]
        w = [f[:, a] if b[a] else 1 - f[:, a] for a in range(3)]
        v = ((n * Z + c[2]) * Y + c[1]) * X + c[0]
        gg.index_add_(0, v, go * (w[0] * w[1] * w[2])[:, None])
        d = (flat[v] * go).sum(1)
        for a in range(3):
            o = [w[e] for e in range(3) if e != a]
            guv[:, a] += d * o[0] * o[1] * (1 if b[a] else -1) * (float(size[a]) - 1) / 2
    return gg.view(N, Z, Y, X, C).permute(0, 4, 1, 2, 3), guv


def rel(a, b):
    return float((a.double() - b).norm() / b.norm().clamp(min=1e-30))


@pytest.mark.parametrize("order", ["rays", "random"])
@pytest.mark.parametrize("C,dims,S,shift", [(8, (11, 11, 11), 1, 0), (8, (17, 17, 17), 127, 0), (8, (2, 5, 3), 4097, 0),
                                            (4, (7, 7, 7), 20003, 0), (12, (5, 4, 6), 3000, 0), (16, (9, 9, 9), 513, 0),
                                            (8, (17, 17, 17), 300001, 0), (8, (9, 9, 9), 70000, 1)])
def test_channels_last_backward(C, dims, S, shift, order):
    print("case: channels-last grid sample backward", C, dims, S, shift, order, flush=True)
    g = torch.Generator(device=DEV).manual_seed(S + C)
    N = 13
    grid = torch.randn(N, *dims, C, device=DEV, generator=g).permute(0, 4, 1, 2, 3)
    uv = torch.rand(S, 3, device=DEV, generator=g) * 2.2 - 1.1
    index = torch.randint(-1, N + 1, (S,), device=DEV, generator=g)
    if order == "rays":  # runs of samples that move slowly through one slot
        t = torch.arange(S, device=DEV)
        index = index[t // 40]
        uv = (uv[t // 40] * 0.5 + (t % 40)[:, None] / 60.0).contiguous()
    gout = torch.randn(S * C + shift, device=DEV, generator=g)[shift:].view(S, C)  # shift: not 16-byte aligned
    assert gout.is_contiguous()
    gg, guv = ops.gs3d_bwd(grid, index, uv, gout)
    rg, ru = reference(grid, index, uv, gout)
    assert rel(gg, rg) <= 1e-6
    assert rel(guv, ru) <= 1e-6
    only, none = ops.gs3d_bwd(grid, index, uv, gout, want_uv=False)
    assert none is None and rel(only, rg) <= 1e-6
