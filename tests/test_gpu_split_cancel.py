"""GPU checks of the FP32 decoder whose hidden biases cancel the sums they are added to (non-negative weights and
activations, the bias minus the mean of the row's sum): its error against FP64 is no larger than that of a plain FP32
evaluation, which rounds the running sum of two products at a time and adds the bias last.

That evaluation is made here step by step from FP32 operands, each step exact in FP64 and rounded once. Nothing else is
allowed for: what the decoder leaves out of a product (2^-26 of it) is a small part of these roundings. (relu only: a silu
of the decoder's has the errors of the hardware exponential, which an evaluation made of torch's functions has not.)"""
import pytest
import torch

from neat_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
S = 50021


def cancelling(H, seed, scale=0.3):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    W0, b0, W1 = rnd(H, 8) / 8 ** 0.5, 0.3 * rnd(H).abs() + 0.5, (rnd(H, H) * (2 / H) ** 0.5).abs()
    W2, b2 = rnd(1, H) * (2 / H) ** 0.5, 0.3 * rnd(1)
    x = scale * rnd(S, 8)
    b1 = -(torch.relu(x @ W0.T + b0) @ W1.T).mean(0)
    return x, (W0, b0, W1, b1, W2, b2)


def fp32_layer(h, W, b):
    """h W^T + b in FP32: two products a step, the bias last."""
    acc = torch.zeros(h.shape[0], W.shape[0], device=DEV)
    H, Wd = h.double(), W.double()
    for k in range(0, W.shape[1], 2):
        acc = (acc.double() + H[:, k:k + 2] @ Wd[:, k:k + 2].T).float()
    return acc + b


@pytest.mark.parametrize("H", [32, 64])
@pytest.mark.parametrize("seed", [0, 1, 2])
def test_forward(seed, H):
    print("case: cancelling decoder, forward", seed, H, flush=True)
    x, p = cancelling(H, seed)
    f = torch.relu
    W0, b0, W1, b1, W2, b2 = (t.double() for t in p)
    want = f(f(x.double() @ W0.T + b0) @ W1.T + b1) @ W2.T + b2
    plain = fp32_layer(f(fp32_layer(f(fp32_layer(x, p[0], p[1])), p[2], p[3])), p[4], p[5])
    packed = torch.cat([t.reshape(-1) for t in p])
    got = ops.decoder_fwd(x, packed, 8, H, 1, 1, "relu", "id", 2.0)
    assert float((got.double() - want).norm()) <= float((plain.double() - want).norm())


@pytest.mark.parametrize("H", [32, 64])
@pytest.mark.parametrize("seed", [0, 1, 2])
def test_output_weight_gradient(seed, H):
    """sum_n h2 dy of output gradients of one sign, against the same sum of the plain evaluation's h2, each product and
    addition rounded (pairwise sums of 2^16 terms: 16 roundings more, 2^-24 of the sum each, sqrt(16) of them allowed for).
    Rows with a unit within rounding of zero are left out: a unit is rounded like its pre-activation there."""
    print("case: cancelling decoder, output weights", seed, H, flush=True)
    x, p = cancelling(H, seed, scale=0.05)
    W0, b0, W1, b1, W2, b2 = (t.double() for t in p)
    z1 = x.double() @ W0.T + b0
    z2 = torch.relu(z1) @ W1.T + b1
    clear = (z1.abs() > 1e-5).all(1) & (z2.abs() > 1e-4).all(1)
    gy = torch.rand(S, 1, device=DEV, generator=torch.Generator(device=DEV).manual_seed(9)) * clear[:, None]
    want = (torch.relu(z2) * gy.double()).sum(0)
    h2 = torch.relu(fp32_layer(torch.relu(fp32_layer(x, p[0], p[1])), p[2], p[3]))
    plain = (h2 * gy).double().sum(0)
    packed = torch.cat([t.reshape(-1) for t in p])
    gp, _ = ops.decoder_bwd(x, packed, gy, 8, H, 1, 1, "relu", "id", 2.0)
    got = gp[-1 - H:-1].double()
    bar = float((plain - want).norm()) + 4 * 2.0 ** -24 * float(want.norm())
    assert float((got - want).norm()) <= bar
