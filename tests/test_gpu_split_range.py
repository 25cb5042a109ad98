"""GPU checks of the FP32 relu decoder's backward on rows with values that its bfloat16 planes cannot take as they are.

Weights and the other rows' inputs sit on coarse dyadic grids, so the masks are known and what is left are FP32 roundings
of the gradient sums: 2^-24 sqrt(n) for n dependent additions, below 1e-6 up to 2^8; 2e-6 is asked for."""
import numpy as np
import pytest
import torch

from neat_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
BAR = 2e-6


def params(H, seed):
    """W in 1/16 steps within +-1/2, those of channel 7 2^-10 times that, no bias zero; as a packed FP32 tensor."""
    g = np.random.default_rng(seed)
    out = []
    for fi, fo in ((8, H), (H, H), (H, 1)):
        w, b = g.integers(-8, 9, (fo, fi)) / 16.0, (2 * g.integers(-4, 4, fo) + 1) / 32.0
        if fi == 8:
            w[:, 7] /= 1024
        out += [w.ravel(), b]
    return torch.from_numpy(np.concatenate(out).astype(np.float32)).to(DEV)


def gradients(x, p, gy, H):
    return ops.decoder_bwd(x, p, gy, 8, H, 1, 1, "relu", "id", 2.0)


@pytest.mark.parametrize("H", [32, 64])
def test_rows_beside_bad_ones(H):
    """A row's infinity, NaN or huge value leaves the input gradients of its tile's other rows alone."""
    print("case: split backward, bad rows", H, flush=True)
    g = torch.Generator(device=DEV).manual_seed(H)
    x = torch.randint(-16, 17, (96, 8), device=DEV, generator=g) / 16.0
    gy = torch.randn(96, 1, device=DEV, generator=g)
    p = params(H, 5)
    clean = gradients(x, p, gy, H)[1].double()
    bad = {3: float("inf"), 17: float("-inf"), 40: float("nan"), 41: 3e38, 42: 3.4e38, 77: 1e35}
    for r, v in bad.items():
        x[r, r % 8] = v
    got = gradients(x, p, gy, H)[1].double()
    keep = [r for r in range(96) if r not in bad]
    assert float((got[keep] - clean[keep]).norm()) <= BAR * float(clean[keep].norm())


@pytest.mark.parametrize("H", [32, 64])
@pytest.mark.parametrize("value", [1e30, 3e38, -3.395e38, 3.4e38])
def test_huge_finite_row(value, H):
    """Where FP32 sums stay finite the gradients are those of FP64: bfloat16 rounds values above 3.39e38 to infinity."""
    print("case: split backward, huge row", value, H, flush=True)
    g = torch.Generator(device=DEV).manual_seed(H)
    x = torch.randint(-16, 17, (96, 8), device=DEV, generator=g) / 16.0
    gy = torch.randn(96, 1, device=DEV, generator=g)
    x[41, 7], gy[41] = value, 2.0 ** -100
    p = params(H, 5)
    P, X = p.double().requires_grad_(True), x.double().requires_grad_(True)
    at, h = 0, X
    for fi, fo in ((8, H), (H, H), (H, 1)):
        h = h @ P[at:at + fi * fo].view(fo, fi).T + P[at + fi * fo:at + fi * fo + fo]
        at += fi * fo + fo
        h = torch.relu(h) if fo != 1 else h
    rp, rx = torch.autograd.grad(h, (P, X), gy.double())
    for a, b in zip(gradients(x, p, gy, H), (rp, rx)):
        assert float((a.double() - b).norm()) <= BAR * float(b.norm())
