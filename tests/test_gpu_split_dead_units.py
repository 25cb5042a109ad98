"""GPU check of the FP32 relu decoder's backward with units that have no weights and no bias (their pre-activation is
exactly zero and relu'(0) = 0, so they neither pass nor get a gradient), in the first, the second and both hidden layers.

The other weights and the inputs sit on coarse dyadic grids, so every mask is known and what is left are FP32 roundings of
the gradient sums: 2^-24 sqrt(n) for n dependent additions, below 1e-6 up to 2^8; 2e-6 is asked for."""
import numpy as np
import pytest
import torch

from neat_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
BAR = 2e-6


@pytest.mark.parametrize("H", [32, 64])
@pytest.mark.parametrize("layers", [(0,), (1,), (0, 1)])
@pytest.mark.parametrize("S", [1, 33, 8193])
def test_units_without_weights(S, layers, H):
    print("case: split decoder, dead units", S, layers, H, flush=True)
    g = np.random.default_rng(S + H)
    blocks = []
    for layer, (fi, fo) in enumerate(((8, H), (H, H), (H, 1))):
        w, b = g.integers(-8, 9, (fo, fi)) / 16.0, (2 * g.integers(-4, 4, fo) + 1) / 32.0
        if layer in layers:
            dead = g.permutation(fo)[:fo - 3]
            w[dead], b[dead] = 0.0, 0.0
        blocks += [w.ravel(), b]
    p = torch.from_numpy(np.concatenate(blocks).astype(np.float32)).to(DEV)
    gen = torch.Generator(device=DEV).manual_seed(S)
    x = torch.randint(-16, 17, (S, 8), device=DEV, generator=gen) / 16.0
    gy = torch.randn(S, 1, device=DEV, generator=gen)
    gp, gx = ops.decoder_bwd(x, p, gy, 8, H, 1, 1, "relu", "id", 2.0)
    P, X = p.double().requires_grad_(True), x.double().requires_grad_(True)
    at, h = 0, X
    for fi, fo in ((8, H), (H, H), (H, 1)):
        h = h @ P[at:at + fi * fo].view(fo, fi).T + P[at + fi * fo:at + fi * fo + fo]
        at += fi * fo + fo
        h = torch.relu(h) if fo != 1 else h
    rp, rx = torch.autograd.grad(h, (P, X), gy.double())
    for a, b in ((gp, rp), (gx, rx)):
        assert float((a.double() - b).norm()) <= BAR * float(b.norm().clamp(min=1e-30))
