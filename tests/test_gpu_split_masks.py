"""GPU check of the relu masks that the FP32 decoder's split backward takes without a plain FP32 evaluation, on random
(not dyadic) decoders, with rows whose units lie as close to zero as any FP32 evaluation can tell.

A sum of n products is off by at most 2 n 2^-24 of the sum A of its terms' magnitudes, however it is ordered and rounded
(n roundings of 2^-23 at most): 10 terms in the first layer, H + 8 in the second (6 partial products down to 2^-18, the
bias), whose inputs bring the first layer's error along. Rows whose units all lie beyond that have masks known from FP64.
A wrong mask moves a row's input gradient by some 10% of a typical row's; 1e-4 of it is asked for."""
import pytest
import torch

from neat_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
U = 2.0 ** -24


@pytest.mark.parametrize("H", [32, 64])
@pytest.mark.parametrize("seed", [0, 1, 2])
def test_masks_near_zero(seed, H):
    print("case: split backward, masks", seed, H, flush=True)
    S = 200003
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    p = (rnd(H, 8) / 8 ** 0.5, 0.3 * rnd(H), rnd(H, H) * (2 / H) ** 0.5, 0.3 * rnd(H), rnd(1, H) * (2 / H) ** 0.5, rnd(1))
    x, gy = rnd(S, 8), 0.5 + torch.rand(S, 1, device=DEV, generator=g)
    W0, b0, W1, b1, W2, _ = (t.double() for t in p)
    X = x.double()
    z1 = X @ W0.T + b0
    e1 = 2 * 10 * U * (X.abs() @ W0.abs().T + b0.abs())
    h1 = torch.relu(z1)
    z2 = h1 @ W1.T + b1
    e2 = e1 @ W1.abs().T + 2 * (H + 8) * U * (h1 @ W1.abs().T + b1.abs())
    known = (z1.abs() > e1).all(1) & (z2.abs() > e2).all(1)
    near = known & ((z1.abs() < 20 * e1).any(1) | (z2.abs() < 20 * e2).any(1))
    assert int(near.sum()) > 1000 and int(known.sum()) > S // 2
    want = (gy.double() * W2 * (z2 > 0)) @ W1 * (z1 > 0) @ W0
    got = ops.decoder_bwd(x, torch.cat([t.reshape(-1) for t in p]), gy, 8, H, 1, 1, "relu", "id", 2.0)[1].double()
    assert float((got - want)[known].norm(dim=1).max()) <= 1e-4 * float(want.norm(dim=1).median())
