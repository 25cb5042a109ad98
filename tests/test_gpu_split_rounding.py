"""GPU check that the rounding of the FP32 relu decoder's backward has no direction: its parameter-gradient sums run on
matrix instructions that round small terms down, so errors would add up over a batch in proportion to its rows, where the
gradient itself (of random signs) grows with their square root.

The mean of (gradient - FP64) over the entries of the hidden layer's weights, in units of their root mean square, with
the rows' factor (the output weight) taken out: errors of 2^-22 an entry (twice what FP32 sums of this length were
measured at), shared along a row at worst, average to 2^-22 / sqrt(H), which is 4.2e-8 for 32 rows; 6e-8 is allowed. A
direction shows at 3e-7 to 4e-7. Rows with a unit within rounding of zero are left out: either mask
would be right there."""
import pytest
import torch

from neat_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("H", [32, 64])
@pytest.mark.parametrize("S", [65536, 300007])
def test_hidden_weight_gradient_has_no_direction(S, H):
    print("case: split decoder, direction of rounding", S, H, flush=True)
    g = torch.Generator(device=DEV).manual_seed(S + H)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    W0, b0, W1, b1 = rnd(H, 8) / 8 ** 0.5, 0.3 * rnd(H), rnd(H, H) * (2 / H) ** 0.5, 0.3 * rnd(H)
    W2 = (0.5 + torch.rand(H, device=DEV, generator=g)) * rnd(H).sign()
    p = torch.cat([t.reshape(-1) for t in (W0, b0, W1, b1, W2, rnd(1))])
    x = rnd(S, 8)
    z1 = x.double() @ W0.double().T + b0.double()
    z2 = torch.relu(z1) @ W1.double().T + b1.double()
    clear = (z1.abs() > 1e-5).all(1) & (z2.abs() > 1e-4).all(1)
    gy = rnd(S, 1) * clear[:, None]
    gp, _ = ops.decoder_bwd(x, p, gy, 8, H, 1, 1, "relu", "id", 2.0)
    at = 8 * H + H
    got = gp[at:at + H * H].view(H, H).double() / W2[:, None].double()
    want = ((z2 > 0) * gy.double()).T @ torch.relu(z1)
    assert abs(float((got - want).mean() / want.square().mean().sqrt())) <= 6e-8
