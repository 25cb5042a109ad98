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


def cancelling(H, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    W0, b0, W1 = rnd(H, 8) / 8 ** 0.5, 0.3 * rnd(H).abs() + 0.5, (rnd(H, H) * (2 / H) ** 0.5).abs()
    W2, b2 = rnd(1, H) * (2 / H) ** 0.5, 0.3 * rnd(1)
    x = 0.3 * rnd(S, 8)
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
