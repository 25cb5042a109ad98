"""GPU check of the FP32 grid-gradient scatter's conversions to fixed point: chunks of at most 64 samples per lane, and a
segment longer than that, whose runs in one cell take the general conversion.

The scatter quantises at 2^-46 of the largest value; what is left are FP32 sums of a cell's run, rounded once per sample.
The runs of the longest segment here hold up to 70 samples and the vector-ALU form it is compared with adds thousands of
samples per vertex in FP32: sqrt(n) 2^-24 with n up to 2^13 is 5e-6. 2e-5 is asked for."""
import pytest
import torch

from neat_amd import ops, pipeline, workloads as W

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("count", [1, 2049, 65536, 65537, 70001])
def test_long_segment(count):
    print("case: grid scatter, first segment's samples", count, flush=True)
    cfg = W.C1
    sc = W.make_scene(cfg, seed=1)
    ds = pipeline.to_device(sc, cfg)
    o, d = W.batch_rays(cfg, 70, seed=3)
    to, td = torch.from_numpy(o).to(DEV), torch.from_numpy(d).to(DEV)
    td[0] = -to[0] / to[0].norm()  # at least one ray through the volume
    segs = dict(pipeline.sample(ds, to, td, jitter=True, seed=2, emit=False))
    n = segs["seg_count"].clone()
    n[0] = count
    segs["seg_count"] = n
    per_ray = torch.zeros(70, dtype=torch.int64, device=DEV).index_add_(0, segs["seg_ray"].long(), n.long())
    segs["ray_sample_offset"] = torch.cat([per_ray.new_zeros(1), per_ray.cumsum(0)])
    gproj = torch.randn(70, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1))
    out = []
    for precision in ("fp32", "fp32_valu"):
        pj = ops.Projector(ds.pos_min, ds.pos_max, ds.prefix, to, td, segs, ds.grid, ds.params, ds.mlp, True, 2,
                           precision=precision)
        pj.forward()
        out.append(pj.backward(gproj)[0].double())
    assert float((out[0] - out[1]).norm() / out[1].norm()) <= 2e-5
