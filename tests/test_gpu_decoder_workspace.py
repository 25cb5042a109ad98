"""GPU check that the standalone decoder's backward stays inside its workspace, whatever number of parameter slices the
batch leaves room for (one per 64 rows, at most 1024): the bytes past the queried size stay as they were, and the
gradients are those of FP64.

Weights and inputs are random and relu units near zero may take either side, so relu rows are compared where every unit
is clear of zero. The sums have at most 2^9 terms, each rounded to 2^-24 a few times: below 3e-6; 1e-5 is asked for."""
import pytest
import torch

from neat_amd import _abi, ops, workloads as W

pytestmark = pytest.mark.gpu
DEV = "cuda"
GUARD = 1 << 18  # bytes past the workspace: more than the slices of a whole workgroup


@pytest.mark.parametrize("H", [32, 64])
@pytest.mark.parametrize("act", ["relu", "silu"])
@pytest.mark.parametrize("S", [1, 64, 65, 128, 129, 192, 193, 256, 257, 511])
def test_slices_stay_in_the_workspace(S, act, H):
    print("case: decoder workspace", S, act, H, flush=True)
    g = torch.Generator(device=DEV).manual_seed(S + H)
    p = torch.from_numpy(W.decoder_params(8, H, 1, 1, 3)).to(DEV)
    x = torch.randn(S, 8, device=DEV, generator=g)
    gy = torch.randn(S, 1, device=DEV, generator=g)
    P, X = p.double().requires_grad_(True), x.double().requires_grad_(True)
    at, h = 0, X
    clear = torch.ones(S, dtype=torch.bool, device=DEV)
    for fi, fo in ((8, H), (H, H), (H, 1)):
        h = h @ P[at:at + fi * fo].view(fo, fi).T + P[at + fi * fo:at + fi * fo + fo]
        at += fi * fo + fo
        if fo != 1:
            clear &= (h.detach().abs() > 1e-5).all(1)
            h = torch.relu(h) if act == "relu" else torch.nn.functional.silu(h)
    if act == "relu":
        gy = gy * clear[:, None]
    rp, rx = torch.autograd.grad(h, (P, X), gy.double())
    n = _abi.lib().neat_decoder_workspace_bytes(S, 8, H, 1, 1)
    buf = torch.full((n + GUARD,), 0xA5, dtype=torch.uint8, device=DEV)
    gp, gx = torch.empty_like(p), torch.empty_like(x)
    _abi.call("neat_decoder_bwd", _abi.stream_ptr(), _abi.ptr(x), S, 8, H, 1, 1, _abi.ptr(p), _abi.ACT[act],
              _abi.ACT["id"], 2.0, _abi.ptr(gy), _abi.ptr(gp), _abi.ptr(gx), _abi.ptr(buf), n)
    assert bool((buf[n:] == 0xA5).all())
    for a, b in ((gp, rp), (gx, rx)):
        assert float((a.double() - b).norm()) <= 1e-5 * float(b.norm().clamp(min=1e-30))
