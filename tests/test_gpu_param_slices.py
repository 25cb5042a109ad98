"""GPU check of the BF16 relu backward's parameter gradient, summed over a workgroup's waves in LDS: both decoder widths,
from a single ray (most workgroups without a chunk) up. Against the FP32 form: 1e-2 for gradients, the bar the BF16
arithmetic is held to against FP64; twice on the same inputs: bit-equal (the sums run in a fixed order)."""
import pytest
import torch

from neat_amd import ops, pipeline, workloads as W

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("H", [32, 64])
@pytest.mark.parametrize("rays", [1, 70, 4001])
def test_bf16_relu_parameter_gradient(rays, H):
    print("case: bf16 relu parameter gradient", rays, H, flush=True)
    cfg = W.C1
    sc = W.make_scene(cfg, seed=1)
    ds = pipeline.to_device(sc, cfg)
    ds.params = torch.from_numpy(W.decoder_params(8, H, 1, 1, 4)).to(DEV)
    ds.mlp = dict(ds.mlp, hidden=H, act="relu")
    o, d = W.batch_rays(cfg, rays, seed=rays)
    to, td = torch.from_numpy(o).to(DEV), torch.from_numpy(d).to(DEV)
    td[0] = -to[0] / to[0].norm()  # at least one ray through the volume
    segs = pipeline.sample(ds, to, td, jitter=True, seed=2, emit=False)
    gproj = torch.randn(rays, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1))
    out = []
    for precision in ("bf16", "bf16", "fp32"):
        pj = ops.Projector(ds.pos_min, ds.pos_max, ds.prefix, to, td, segs, ds.grid, ds.params, ds.mlp, True, 2,
                           precision=precision)
        pj.forward()
        out.append(pj.backward(gproj)[1].double())
    assert torch.equal(out[0], out[1])
    assert float((out[0] - out[2]).norm() / out[2].norm()) <= 1e-2
