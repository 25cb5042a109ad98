"""GPU checks of the FP32 decoder in split form (three BF16 planes per FP32 value), standalone and in the projector, at
the edges of its tiles.

Weights and inputs sit on coarse dyadic grids, so every pre-activation is exact in FP32 in any order of additions: many
units are exactly zero, the relu masks are known, and what is left are the FP32 roundings of the gradient sums. A
result of n additions with rounding 2^-24 stays within 2^-24 sqrt(n) (norm-wise), here below 1e-6 for up to 2^8
dependent additions; 2e-6 is asked for."""
import numpy as np
import pytest
import torch

from neat_amd import ops, pipeline, workloads as W

pytestmark = pytest.mark.gpu
DEV = "cuda"
BAR = 2e-6


def dyadic_params(H, seed):
    """W in 1/16 steps within +-1/2 (a fifth of them zero), biases in 1/16 steps, packed."""
    g = np.random.default_rng(seed)
    out = []
    for fi, fo in ((8, H), (H, H), (H, 1)):
        w = g.integers(-8, 9, fo * fi) / 16.0
        out += [w * (g.random(w.size) > 0.2), g.integers(-4, 5, fo) / 16.0]
    return torch.from_numpy(np.concatenate(out).astype(np.float32)).to(DEV)


def reference(x, params, H, act, last_act, gy):
    P = params.double().requires_grad_(True)
    X = x.double().requires_grad_(True)
    at, h = 0, X
    for fi, fo in ((8, H), (H, H), (H, 1)):
        h = h @ P[at:at + fi * fo].view(fo, fi).T + P[at + fi * fo:at + fi * fo + fo]
        at += fi * fo + fo
        if fo != 1:
            h = torch.relu(h) if act == "relu" else torch.nn.functional.silu(h)
    y = torch.nn.functional.softplus(h, beta=2.0, threshold=20) if last_act == "softplus" else h
    gp, gx = torch.autograd.grad(y, (P, X), gy.double())
    return y.detach(), gp, gx


def rel(a, b):
    return float((a.double() - b).norm() / b.norm().clamp(min=1e-30))


@pytest.mark.parametrize("H", [32, 64])
@pytest.mark.parametrize("act,last_act", [("relu", "softplus"), ("relu", "id"), ("silu", "softplus")])
@pytest.mark.parametrize("S", [1, 31, 33, 256, 8193, 200003])
def test_decoder_edges(S, act, last_act, H):
    print("case: split decoder", S, act, last_act, H, flush=True)
    g = torch.Generator(device=DEV).manual_seed(S + H)
    x = torch.randint(-16, 17, (S, 8), device=DEV, generator=g) / 16.0
    gy = torch.randn(S, 1, device=DEV, generator=g)
    p = dyadic_params(H, S)
    y = ops.decoder_fwd(x, p, 8, H, 1, 1, act, last_act, 2.0)
    gp, gx = ops.decoder_bwd(x, p, gy, 8, H, 1, 1, act, last_act, 2.0)
    ry, rp, rx = reference(x, p, H, act, last_act, gy)
    assert rel(y, ry) <= BAR
    assert rel(gx, rx) <= BAR
    assert rel(gp, rp) <= BAR


@pytest.mark.parametrize("H", [32, 64])
def test_decoder_outside_the_split_range(H):
    """Rows with infinities, NaN and huge values give what plain FP32 arithmetic gives (relu maps NaN to 0, as
    x > 0 ? x : 0 does) and leave the other rows of their tile alone."""
    print("case: split decoder, non-finite rows", H, flush=True)
    g = torch.Generator(device=DEV).manual_seed(H)
    x = torch.randint(-16, 17, (96, 8), device=DEV, generator=g) / 16.0
    clean = x.clone()
    bad = {3: float("inf"), 17: float("-inf"), 40: float("nan"), 41: 3e38, 77: 1e35}
    for r, v in bad.items():
        x[r, r % 8] = v
    p = dyadic_params(H, 5)
    y = ops.decoder_fwd(x, p, 8, H, 1, 1, "relu", "id", 2.0).cpu()
    yc = ops.decoder_fwd(clean, p, 8, H, 1, 1, "relu", "id", 2.0).cpu()
    keep = [r for r in range(96) if r not in bad]
    assert rel(y[keep], yc[keep].double()) <= BAR
    h, at, pc = x.cpu(), 0, p.cpu()
    for fi, fo in ((8, H), (H, H), (H, 1)):
        w, b = pc[at:at + fi * fo].view(fo, fi), pc[at + fi * fo:at + fi * fo + fo]
        h = (h[:, None, :] * w[None]).sum(2) + b
        at += fi * fo + fo
        if fo != 1:
            h = torch.where(h > 0, h, torch.zeros_like(h))
    for r in bad:
        assert torch.isnan(y[r]) == torch.isnan(h[r]) and torch.isposinf(y[r]) == torch.isposinf(h[r])
        if torch.isfinite(h[r]):
            assert abs(y[r] - h[r]) <= 1e-5 * abs(h[r])


@pytest.mark.parametrize("H,act", [(32, "relu"), (64, "relu"), (64, "silu")])
@pytest.mark.parametrize("rays", [1, 3, 70, 4001])
def test_projector_against_vector_form(rays, H, act):
    """The FP32 projector against the vector-ALU form (the same sample positions and masks, plain FP32 sums)."""
    print("case: split projector", rays, H, act, flush=True)
    cfg = W.C1
    sc = W.make_scene(cfg, seed=1)
    ds = pipeline.to_device(sc, cfg)
    ds.grid.copy_((ds.grid * 160).round() / 64)  # features on a grid; trilinear weights round both forms alike
    ds.params = dyadic_params(H, 3)
    ds.params[:8 * H] += 1.0 / 64  # no pre-activation exactly at zero: positions carry rounding
    ds.mlp = dict(ds.mlp, hidden=H, act=act)
    o, d = W.batch_rays(cfg, rays, seed=rays)
    to, td = torch.from_numpy(o).to(DEV), torch.from_numpy(d).to(DEV)
    td[0] = -to[0] / to[0].norm()  # at least one ray through the volume
    segs = pipeline.sample(ds, to, td, jitter=True, seed=2, emit=False)
    gproj = torch.randn(rays, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1))
    out = []
    for precision in ("fp32", "fp32_valu"):
        pj = ops.Projector(ds.pos_min, ds.pos_max, ds.prefix, to, td, segs, ds.grid, ds.params, ds.mlp, True, 2,
                           precision=precision)
        out.append([pj.forward(), *pj.backward(gproj)])
    for a, b in zip(*out):
        assert rel(a, b.double()) <= 1e-5  # both within 1e-5 of the oracle's FP32 form; a unit at zero may flip


@pytest.mark.parametrize("H", [32, 64])
@pytest.mark.parametrize("rays", [1, 3, 70, 4001])
def test_bf16_silu_projector_edges(rays, H):
    """The BF16 form with silu against the FP32 form: 1e-3 for projections and 1e-2 for gradients, the bars the BF16
    arithmetic is held to against FP64."""
    print("case: bf16 silu projector", rays, H, flush=True)
    cfg = W.C1
    sc = W.make_scene(cfg, seed=1)
    ds = pipeline.to_device(sc, cfg)
    ds.params = torch.from_numpy(W.decoder_params(8, H, 1, 1, 4)).to(DEV)
    ds.mlp = dict(ds.mlp, hidden=H, act="silu")
    o, d = W.batch_rays(cfg, rays, seed=rays)
    to, td = torch.from_numpy(o).to(DEV), torch.from_numpy(d).to(DEV)
    td[0] = -to[0] / to[0].norm()  # at least one ray through the volume
    segs = pipeline.sample(ds, to, td, jitter=True, seed=2, emit=False)
    gproj = torch.randn(rays, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1))
    out = []
    for precision in ("bf16", "fp32"):
        pj = ops.Projector(ds.pos_min, ds.pos_max, ds.prefix, to, td, segs, ds.grid, ds.params, ds.mlp, True, 2,
                           precision=precision)
        out.append([pj.forward(), *pj.backward(gproj)])
    for a, b, bar in zip(*out, (1e-3, 1e-2, 1e-2)):
        assert rel(a, b.double()) <= bar
