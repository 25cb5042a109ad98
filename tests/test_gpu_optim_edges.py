"""GPU checks of the optimizer's vector kernels at their edges: Adam's four-at-a-time form and the eight-at-a-time BF16
copy with remainders and (for the copy) unaligned arrays. Adam is held to the same operations one by one in float64
(a handful of FP32 roundings: 1e-6 of the values), the copy to round-to-nearest-even bit for bit."""
import pytest
import torch

from neat_amd import _abi, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 1025, 17_000_003])
@pytest.mark.parametrize("wd", [0.0, 0.01])
def test_adam_remainders(n, wd):
    print("case: adam", n, wd, flush=True)
    g = torch.Generator(device=DEV).manual_seed(n)
    p, gr, m = (torch.randn(n, device=DEV, generator=g) for _ in range(3))
    v = torch.rand(n, device=DEV, generator=g)
    P, G, M, V = (t.double() for t in (p, gr, m, v))
    ops.adam_step(p, gr, m, v, 1e-2, 9, weight_decay=wd)
    G = G + wd * P
    M = 0.9 * M + 0.1 * G
    V = 0.999 * V + 0.001 * G * G
    P = P - 1e-2 / (1 - 0.9 ** 9) * M / (V.sqrt() / (1 - 0.999 ** 9) ** 0.5 + 1e-8)
    for a, b in ((p, P), (m, M), (v, V)):
        assert float((a.double() - b).abs().max()) <= 1e-6 * float(b.abs().max())


@pytest.mark.parametrize("n", [1, 7, 8, 9, 2047, 2049, 100_001])
@pytest.mark.parametrize("shift", [0, 1])
def test_bf16_copy_remainders(n, shift):
    print("case: bf16 copy", n, shift, flush=True)
    x = torch.randn(n + shift, device=DEV, generator=torch.Generator(device=DEV).manual_seed(n))[shift:]
    out = torch.full((n + 16,), 7, dtype=torch.int16, device=DEV)
    _abi.call("neat_grid_to_bf16", _abi.stream_ptr(), _abi.ptr(x), n, _abi.ptr(out))
    assert torch.equal(out[:n], x.to(torch.bfloat16).view(torch.int16))
    assert bool((out[n:] == 7).all())
