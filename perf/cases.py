"""Performance cases of the projector framework, through its Python entry points (neat_amd.ops, neat_amd.pipeline,
neat_amd.proposal): the calls that a reconstruction program makes, from a few hundred rays to full 2^18-ray batches.

Scenes are the two geometries of the projector benchmark suite: "small" (uniform depth-2 octree, 64 leaves, 11^3 x 8
grids, decoder 8->32->32->1, at most 32 samples per node, 128^2 detector) and "full" (depth-5 octree refined where a
100-ellipsoid phantom varies, 4096 leaves, 17^3 x 8 grids, decoder 8->64->64->1, at most 64 samples per node, 512^2
detector). Kinds of case:

  view   projections only (rendering a view, validation): sample the rays, plan, forward. No jitter.
  step   one training step's forward and backward: sample (jittered), plan, forward, FP64 MSE, backward to grid and
         decoder; optionally the gradient onto the rays (pose refinement) or the learned proposal's placement.
  gather the indirect trilinear grid sample used on its own (IndirectGridSample3D), forward and backward with uv
         gradients, at the samples of a batch of rays.
  mlp    the decoder used on its own (FCBlock and the output activation), forward and backward.
  reg    the volume regulariser of a training step: total variation and edge loss with the grid gradient.
  adam   the optimizer's step on the grid and the decoder, and the refresh of the grid's BF16 copy.

Everything but `prepare` and `run` is plain torch / numpy: `exact` restates the paths in 64 bits (the segments, whose
sample counts are steps in FP32, with the FP32 operations that define them).
"""
import functools
import heapq
import math

import numpy as np
import torch

from neat_amd import ops, pipeline, proposal

SCENES = {
    # samples_per_ray: the mean over the detector (uniform samples, proposal samples), for work()
    "small": dict(depth=2, leaves=0, G=11, H=32, views=256, det=128, spn=32, ellipsoids=20, samples_per_ray=(37, 25)),
    "full": dict(depth=5, leaves=4096, G=17, H=64, views=256, det=512, spn=64, ellipsoids=100,
                 samples_per_ray=(204, 124)),
}
C = 8  # feature channels
BETA = 2.0  # softplus of the decoder's output


def listed():
    return [
        # a thumbnail of a view while reconstructing: the smallest call, launches and host work
        dict(name="view_small_fp32_509", kind="view", scene="small", rays=509, precision="fp32", act="relu"),
        # a full 512 x 512 view of the reconstruction, the inference form
        dict(name="view_full_bf16", kind="view", scene="full", rays=512 * 512, precision="bf16", act="relu"),
        # training on the small scene with an odd, small batch, the default precision
        dict(name="step_small_fp32_4099", kind="step", scene="small", rays=4099, precision="fp32", act="relu",
             pose=False, proposal=False),
        # training on the small scene at the benchmark's batch
        dict(name="step_small_bf16", kind="step", scene="small", rays=1 << 18, precision="bf16", act="relu",
             pose=False, proposal=False),
        # training on the full scene at the benchmark's batch in the default precision (the largest)
        dict(name="step_full_fp32", kind="step", scene="full", rays=1 << 18, precision="fp32", act="relu",
             pose=False, proposal=False),
        # the headline training step: BF16 with the learned proposal
        dict(name="step_full_bf16_proposal", kind="step", scene="full", rays=1 << 18, precision="bf16", act="relu",
             pose=False, proposal=True),
        # a decoder with smooth hidden activations, an odd batch
        dict(name="step_full_bf16_silu_50021", kind="step", scene="full", rays=50021, precision="bf16", act="silu",
             pose=False, proposal=False),
        # pose refinement: gradients onto the rays as well
        dict(name="step_full_fp32_pose_32771", kind="step", scene="full", rays=32771, precision="fp32", act="relu",
             pose=True, proposal=False),
        # the module API's grid sample at the samples of about 2^16 rays
        dict(name="gather_full_13000003", kind="gather", scene="full", samples=13000003),
        # the module API's decoder on a million feature vectors
        dict(name="mlp_relu64_1000003", kind="mlp", rows=1000003, hidden=64, act="relu"),
        # the regulariser of every training step of the full scene
        dict(name="reg_full", kind="reg", scene="full", leaves=4096),
        # the optimizer of every training step of the full scene
        dict(name="adam_full", kind="adam", slots=4096, G=17, hidden=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["view", "step", "step", "step", "gather", "mlp", "reg", "adam"])
    if kind == "mlp":
        return dict(kind=kind, rows=_log_int(rng, 1000, 4_000_000), hidden=rng.choice([32, 64]),
                    act=rng.choice(["relu", "silu"]))
    if kind == "reg":
        return dict(kind=kind, scene="full", leaves=1 + 7 * _log_int(rng, 9, 585))
    if kind == "adam":
        return dict(kind=kind, slots=_log_int(rng, 64, 4096), G=rng.choice([9, 11, 13, 17]),
                    hidden=rng.choice([32, 64]))
    scene = rng.choice(["small", "full"])
    if kind == "gather":
        return dict(kind=kind, scene=scene, samples=_log_int(rng, 10000, 13_000_000 if scene == "full" else 2_500_000))
    precision = rng.choice(["fp32", "bf16"])
    case = dict(kind=kind, scene=scene, rays=_log_int(rng, 200, 1 << 18), precision=precision,
                act=rng.choice(["relu", "relu", "silu"]))
    if kind == "step":
        case["pose"] = rng.random() < 0.25
        case["proposal"] = precision == "bf16" and case["act"] == "relu" and rng.random() < 0.5
    return case


# ---- inputs (plain numpy / torch) -------------------------------------------------------------------------------------
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


@functools.lru_cache(maxsize=None)
def _boxes(depth):
    """Boxes and depths of the complete octree of [-1, 1]^3, numbered breadth first (child i of n is 8n + 1 + i and
    takes the upper half on axis k iff bit k of i is set)."""
    mn, mx, dep = [np.full((1, 3), -1.0)], [np.full((1, 3), 1.0)], [np.zeros(1, np.int32)]
    bits = (np.arange(8)[:, None] >> np.arange(3)) & 1
    for d in range(depth):
        c = (mn[-1] + mx[-1]) / 2
        lo = np.where(bits[None] == 1, c[:, None], mn[-1][:, None])
        hi = np.where(bits[None] == 1, mx[-1][:, None], c[:, None])
        mn.append(lo.reshape(-1, 3))
        mx.append(hi.reshape(-1, 3))
        dep.append(np.full(8 ** (d + 1), d + 1, np.int32))
    return (np.concatenate(mn).astype(np.float32), np.concatenate(mx).astype(np.float32), np.concatenate(dep))


@functools.lru_cache(maxsize=None)
def _tree(name, leaves):
    """The octree of a scene: boxes, 0/1 active flags, active ids (ascending) and the node -> slot table. Adaptive
    scenes split the leaf where the phantom's density varies most (times its edge) until `leaves`."""
    sc = SCENES[name]
    pmin, pmax, dep = _boxes(sc["depth"])
    active = np.zeros(len(dep), np.int32)
    if not leaves:
        active[dep == sc["depth"]] = 1
    else:
        g = np.random.default_rng(11)
        pts = (np.arange(4) + 0.5) / 4
        lat = np.stack(np.meshgrid(pts, pts, pts, indexing="ij"), -1).reshape(-1, 3)
        p = torch.as_tensor(pmin[:, None] + lat * (pmax - pmin)[:, None], dtype=torch.float64, device=_dev())
        rho = torch.zeros(p.shape[:2], dtype=torch.float64, device=p.device)
        for _ in range(sc["ellipsoids"]):
            cen, ax, val = g.uniform(-0.6, 0.6, 3), g.uniform(0.05, 0.35, 3), g.uniform(0, 1)
            q = (p - torch.as_tensor(cen, device=p.device)) / torch.as_tensor(ax, device=p.device)
            rho += val * ((q * q).sum(-1) <= 1)
        score = (rho.std(1, unbiased=False).cpu().numpy() * (pmax - pmin)[:, 0] + 1e-9 * (sc["depth"] - dep)).round(9)
        active[0], heap, n = 1, [(-score[0], 0)], 1
        while heap and n + 7 <= leaves:
            k = heapq.heappop(heap)[1]
            active[k] = 0
            for c in range(8 * k + 1, 8 * k + 9):
                active[c] = 1
                if dep[c] < sc["depth"]:
                    heapq.heappush(heap, (-score[c], c))
            n += 7
    ids = np.flatnonzero(active).astype(np.int64)
    prefix = np.full(len(dep), -1, np.int64)
    prefix[ids] = np.arange(len(ids))
    return dict(pmin=pmin, pmax=pmax, active=active, ids=ids, prefix=prefix, depth=sc["depth"])


def _gen(seed, what):
    return torch.Generator(device=_dev()).manual_seed(1000003 * int(seed) + what)


def _grid(slots, G, seed):
    """Features of a field in training, channels-last in memory."""
    return (torch.randn(slots, G, G, G, C, device=_dev(), generator=_gen(seed, 1)) * 0.1).permute(0, 4, 1, 2, 3)


def _params(hidden, seed):
    """Packed decoder parameters (W [out, in], b per layer): Xavier-uniform weights, biases in +-1 / sqrt(in)."""
    g = np.random.default_rng([int(seed), 2])
    out = []
    for fi, fo in ((C, hidden), (hidden, hidden), (hidden, 1)):
        a = math.sqrt(6.0 / (fi + fo))
        out += [g.uniform(-a, a, fo * fi), g.uniform(-1 / math.sqrt(fi), 1 / math.sqrt(fi), fo)]
    return torch.from_numpy(np.concatenate(out).astype(np.float32)).to(_dev())


def _rays(case, seed):
    """Cone-beam rays (source at distance 4, detector of +-3 on the other side): consecutive pixels for a view, pixels
    drawn over all views and sorted for a step. Origin and unit direction, float32 [R, 3]."""
    sc = SCENES[case["scene"]]
    V, D, R = sc["views"], sc["det"], case["rays"]
    g = _gen(seed, 3)
    if case["kind"] == "view":
        first = torch.randint(0, V * D * D - R + 1, (1,), device=_dev(), generator=g)
        if R >= D * D:
            first = first // (D * D) * (D * D)  # whole views
        idx = first + torch.arange(R, device=_dev())
    else:
        idx = torch.randint(0, V * D * D, (R,), device=_dev(), generator=g).sort().values
    th = 2 * math.pi * (idx // (D * D)).double() / V
    u = ((idx % D).double() + 0.5) / D * 6 - 3
    v = ((idx // D % D).double() + 0.5) / D * 6 - 3
    s, c, z = torch.sin(th), torch.cos(th), torch.zeros_like(th)
    src = 4 * torch.stack([-s, -c, z], 1)
    d = -2 * src + torch.stack([u * c, -u * s, -v], 1)
    d = d / d.norm(dim=1, keepdim=True)
    return src.float().contiguous(), d.float().contiguous()


def _proposal_inputs(case, seed, slots):
    """Network parameters and a roughness table with the tiers of a trained field (about a third of the slots smooth,
    half in the middle tier, the rest rough)."""
    g = np.random.default_rng([int(seed), 4])
    out = []
    for fi, fo in ((6, 32), (32, 32), (32, 8)):
        a = math.sqrt(6.0 / (fi + fo))
        out += [g.uniform(-a, a, fo * fi), g.uniform(-0.1, 0.1, fo)]
    params = torch.from_numpy(np.concatenate(out).astype(np.float32)).to(_dev())
    rough = torch.from_numpy(np.exp(g.normal(-0.6, 1.2, slots)).astype(np.float32)).to(_dev())
    return params, rough


TAU, TAU_UNIFORM, SHORT, MID = 0.3, 2.0, 8, 24  # tiers of the proposal gate, samples of the smooth and middle tier


def _inputs(case, seed):
    kind, dev = case["kind"], _dev()
    if kind == "mlp":
        H = case["hidden"]
        return dict(x=torch.randn(case["rows"], C, device=dev, generator=_gen(seed, 5)) * 0.3,
                    gy=torch.randn(case["rows"], 1, device=dev, generator=_gen(seed, 6)), params=_params(H, seed))
    if kind == "adam":
        grid, params = _grid(case["slots"], case["G"], seed), _params(case["hidden"], seed)
        like = lambda k, t, s: torch.randn(t.numel(), device=dev, generator=_gen(seed, k)) * s  # noqa: E731
        out = dict(step=7 + seed % 50)
        for n, t in (("grid", grid), ("params", params)):
            lay = (lambda f: f.view(t.shape[0], *t.shape[2:], C).permute(0, 4, 1, 2, 3)) if t.dim() == 5 else \
                (lambda f: f)
            k = 10 if n == "grid" else 20
            out[n] = [t, lay(like(k, t, 1e-3)), lay(like(k + 1, t, 1e-3)), lay(like(k + 2, t, 1e-3).square())]
        return out
    sc = SCENES[case["scene"]]
    tree = _tree(case["scene"], case.get("leaves", sc["leaves"]))
    out = dict(tree=tree, sc=sc, seed=int(seed) % 65521 + 1, grid=_grid(len(tree["ids"]), sc["G"], seed),
               params=_params(sc["H"], seed))
    if kind == "reg":
        return out
    if kind == "gather":
        # the first samples of somewhat more rays than hold them
        case = dict(case, rays=int(case["samples"] / sc["samples_per_ray"][0] * 1.2) + 600)
    out["o"], out["d"] = _rays(case, seed)
    out["target"] = torch.rand(case["rays"], device=dev, generator=_gen(seed, 7))
    if case.get("proposal"):
        out["proposal"] = _proposal_inputs(case, seed, len(tree["ids"]))
    if kind == "gather":
        g = _segments(case, out)
        seg, t, _ = _samples(case, out, g, 0, len(g["n"]), True)
        seg, t = seg[:case["samples"]], t[:case["samples"]]
        p = out["o"].double()[g["ray"][seg]] + out["d"].double()[g["ray"][seg]] * t[:, None]
        slot = g["slot"][seg]
        out["uv"] = ((p - g["mn"][slot]) / (g["mx"][slot] - g["mn"][slot]) * 2 - 1).float()
        out["slot"] = slot
        out["gout"] = torch.randn(len(slot), C, device=dev, generator=_gen(seed, 8))
    return out


# ---- the framework's path ---------------------------------------------------------------------------------------------
def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = dict(case)
    kind = case["kind"]
    if kind == "adam":
        s["bf16"] = ops.grid_to_bf16(s["grid"][0])
    if kind in ("mlp", "adam", "gather"):
        return s
    t, sc = s["tree"], s["sc"]
    dev = _dev()
    mlp = dict(**{"in": C}, hidden=sc["H"], layers=1, out=1, act=case.get("act", "relu"), last_act="softplus",
               beta=BETA)
    s["ds"] = ds = pipeline.DeviceScene(
        max_depth=t["depth"], pos_min=torch.from_numpy(t["pmin"]).to(dev), pos_max=torch.from_numpy(t["pmax"]).to(dev),
        flags=ops.tree_flags(t["active"], t["depth"]).to(dev), prefix=torch.from_numpy(t["prefix"]).to(dev),
        grid=s["grid"], params=s["params"], mlp=mlp, max_spn=sc["spn"])
    s["ids"] = torch.from_numpy(t["ids"]).to(dev)
    if case.get("precision") == "bf16":
        s["bf16"] = ops.grid_to_bf16(ds.grid)  # a training program refreshes this copy in its optimizer step
    if case.get("proposal"):
        p = proposal.ProposalSampler(dev, num_samples=SHORT, num_slots=ds.grid.shape[0], tau=TAU,
                                     tau_uniform=TAU_UNIFORM, mid_samples=MID)
        p.params, p.roughness = s["proposal"]
        s["proposal"] = p
    return s


def _projector(s, jitter):
    c, ds = s["case"], s["ds"]
    segs = pipeline.sample(ds, s["o"], s["d"], jitter=jitter, seed=s["seed"], emit=False)
    if c.get("proposal"):
        segs = s["proposal"].apply(s["o"], s["d"], segs, ds.prefix)
    return ops.Projector(ds.pos_min, ds.pos_max, ds.prefix, s["o"], s["d"], segs, ds.grid, ds.params, ds.mlp, jitter,
                         s["seed"], precision=c["precision"], grid_bf16=s.get("bf16"))


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "view":
        return {"proj": _projector(s, False).forward()}
    if kind == "step":
        pj = _projector(s, True)
        proj = pj.forward()
        _, gproj = ops.mse_fp64(proj, s["target"])
        out = {"proj": proj}
        out["grid"], out["params"] = pj.backward(gproj)
        if c["pose"]:
            out["origin"], out["direction"] = pj.ray_grad()
        return out
    if kind == "gather":
        feat = ops.gs3d_fwd(s["grid"], s["slot"], s["uv"])
        gg, guv = ops.gs3d_bwd(s["grid"], s["slot"], s["uv"], s["gout"])
        return {"feat": feat, "grid": gg, "uv": guv}
    if kind == "mlp":
        dims = (C, c["hidden"], 1, 1, c["act"], "softplus", BETA)
        y = ops.decoder_fwd(s["x"], s["params"], *dims)
        gp, gx = ops.decoder_bwd(s["x"], s["params"], s["gy"], *dims)
        return {"y": y, "params": gp, "x": gx}
    if kind == "reg":
        ds = s["ds"]
        loss, gg = ops.volume_regularizer(ds.pos_min, ds.pos_max, ds.flags, ds.prefix, s["ids"], ds.grid,
                                          seed=s["seed"])
        return {"loss": loss, "grid": gg}
    p, g, m, v = s["grid"]
    ops.adam_step(p, g, m, v, 1e-2, s["step"])
    q = s["params"]
    ops.adam_step(*q, 1e-3, s["step"])
    ops.grid_to_bf16(p, out=s["bf16"])
    return {"grid": p, "m": m, "v": v, "bf16": s["bf16"], "params": q[0], "pm": q[2], "pv": q[3]}


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "mlp":
        H, n = case["hidden"], case["rows"]
        return {"bytes": 4 * n * (2 * C + 2), "flops": 3 * n * 2 * (C * H + H * H + H)}
    if kind == "adam":
        n = case["slots"] * case["G"] ** 3 * C
        return {"bytes": n * 30, "flops": n * 12}
    sc = SCENES[case["scene"]]
    slots = case.get("leaves", sc["leaves"]) or 8 ** sc["depth"]
    grid = slots * sc["G"] ** 3 * C * 4
    if kind == "reg":
        return {"bytes": 2 * grid, "flops": grid / 4 * 12}
    R = case.get("rays", 0)
    S = case.get("samples") or R * sc["samples_per_ray"][1 if case.get("proposal") else 0]
    if kind == "gather":
        # no more of the grid is read than the samples' corners
        return {"bytes": min(grid, S * 8 * C * 4) + grid + S * (8 + 12 + 2 * C * 4 + 12), "flops": S * C * 8 * 8}
    mlp = 2 * (C * sc["H"] + sc["H"] ** 2 + sc["H"])
    read = min(grid, S * 8 * C * 4) / (2 if case["precision"] == "bf16" else 1)
    if kind == "view":
        return {"bytes": read + R * 28, "flops": S * (mlp + 16 * C)}
    return {"bytes": read + grid + R * (36 + (24 if case["pose"] else 0)), "flops": S * (3 * mlp + 32 * C)}


# ---- the same in 64 bits -------------------------------------------------------------------------------------------------
def _i64(v):
    return v - (1 << 64) if v >= 1 << 63 else v


def _shr(z, k):
    return (z >> k) & ((1 << (64 - k)) - 1)


def _mix64(z):
    z = (z ^ _shr(z, 30)) * _i64(0xBF58476D1CE4E5B9)
    z = (z ^ _shr(z, 27)) * _i64(0x94D049BB133111EB)
    return z ^ _shr(z, 31)


def _unit24(h):
    return (_shr(h, 40)).double() / 16777216.0


_GOLD = _i64(0x9E3779B97F4A7C15)


def _segments(case, s):
    """Leaf segments of every ray in (ray, tmin, node) order: the slab test and the sample count in FP32, as the
    framework defines them."""
    t, sc, o, d = s["tree"], s["sc"], s["o"], s["d"]
    dev = o.device
    ids = torch.from_numpy(t["ids"]).to(dev)
    mn, mx = torch.from_numpy(t["pmin"]).to(dev)[ids], torch.from_numpy(t["pmax"]).to(dev)[ids]
    e = mx - mn
    diag = torch.sqrt(e[:, 0] * e[:, 0] + (e[:, 1] * e[:, 1] + e[:, 2] * e[:, 2]))
    parts = []
    step = max(1, (1 << 25) // len(ids))
    for r0 in range(0, o.shape[0], step):
        oo, dd = o[r0:r0 + step], d[r0:r0 + step]
        near = torch.full((oo.shape[0], len(ids)), -236436436.0, device=dev)
        far = torch.full_like(near, 43637575.0)
        hit = torch.ones_like(near, dtype=torch.bool)
        for k in range(3):
            ok, dk = oo[:, k:k + 1], dd[:, k:k + 1]
            zero = dk == 0
            a, b = (mn[None, :, k] - ok) / dk, (mx[None, :, k] - ok) / dk
            lo, hi = torch.minimum(a, b), torch.maximum(a, b)
            near = torch.where(zero, near, torch.maximum(near, lo))
            far = torch.where(zero, far, torch.minimum(far, hi))
            hit &= ~(zero & ((ok < mn[None, :, k]) | (ok >= mx[None, :, k])))
        hit &= (near <= far) & (far >= 0) & ~((far - near).double() < 1e-5)
        r, a = torch.nonzero(hit, as_tuple=True)
        parts.append((r + r0, a, near[r, a], far[r, a]))
    ray, slot, tmin, tmax = (torch.cat(x) for x in zip(*parts))
    # rows are in (ray, slot) order and slots ascend with the node id: one stable sort by tmin inside the rays
    order = tmin.argsort(stable=True)
    order = order[ray[order].argsort(stable=True)]
    ray, slot, tmin, tmax = ray[order], slot[order], tmin[order], tmax[order]
    first = torch.searchsorted(ray, torch.arange(o.shape[0], device=dev))
    rank = torch.arange(len(ray), device=dev) - first[ray]
    n = torch.ceil((tmax - tmin) / diag[slot] * float(sc["spn"])).long()
    return dict(ray=ray, slot=slot, tmin=tmin.double(), tmax=tmax.double(), rank=rank, n=n, mn=mn.double(),
                mx=mx.double())


def _proposal64(s, g):
    """Sample counts and CDF rows (zero: uniform) of the gated proposal, the network in 64 bits."""
    params, rough = s["proposal"]
    o, d = s["o"].double()[g["ray"]], s["d"].double()[g["ray"]]
    h, at = torch.cat([o + d * g["tmin"][:, None], o + d * g["tmax"][:, None]], 1), 0
    for i, (fi, fo) in enumerate(((6, 32), (32, 32), (32, 8))):
        w = params[at:at + fi * fo].double().view(fo, fi)
        b = params[at + fi * fo:at + fi * fo + fo].double()
        at += fi * fo + fo
        h = h @ w.T + b
        h = h.clamp(min=0) if i < 2 else h
    cdf = torch.cumsum(0.75 * torch.softmax(h, 1) + 0.25 / 8, 1)
    cdf[:, 7] = 1.0
    r, n = rough[g["slot"]], g["n"]
    count = torch.where(r <= TAU, n.clamp(max=SHORT), torch.where(r <= TAU_UNIFORM, n.clamp(max=MID), n))
    use = (n > SHORT) & (r <= TAU_UNIFORM)
    return torch.where(use, count, n), torch.where(use[:, None], cdf, torch.zeros_like(cdf))


def _samples(case, s, g, k0, k1, jitter):
    """The samples of segments [k0, k1): segment, t, weight."""
    n = g["n"][k0:k1]
    seg = torch.repeat_interleave(torch.arange(k0, k1, device=n.device), n)
    j = torch.arange(len(seg), device=n.device) - torch.repeat_interleave(torch.cumsum(n, 0) - n, n)
    nn, lo, hi = g["n"][seg].double(), g["tmin"][seg], g["tmax"][seg]

    def place(jj):
        if not jitter:
            return 0.5
        h = _mix64(torch.tensor(s["seed"], device=n.device) ^ (g["ray"][seg] * _GOLD))
        return _unit24(_mix64(h ^ ((g["rank"][seg] << 32) | (jj & 0xFFFFFFFF))))

    def at(jj):
        a, step = place(jj), (hi - lo) / nn
        return (lo + jj * step) * (1 - a) + (lo + (jj + 1) * step) * a

    t = at(j)
    left = torch.where(j == 0, lo, 0.5 * (at(j - 1) + t))
    right = torch.where(j == g["n"][seg] - 1, hi, 0.5 * (at(j + 1) + t))
    w = right - left
    if "cdf" in g:
        c = g["cdf"][seg]
        zero = torch.zeros_like(c[:, :1])

        def cell(jj):
            u = (jj.double() / nn)[:, None]
            b = (c[:, :7] <= u).sum(1, keepdim=True)
            below, above = torch.cat([zero, c], 1).gather(1, b), c.gather(1, b)
            f = ((u - below) / (above - below).clamp(min=1e-300)).clamp(0, 1)
            x = lo + (hi - lo) * ((b + f) * 0.125)[:, 0]
            return torch.where(jj <= 0, lo, torch.where(jj >= g["n"][seg], hi, x))

        use = c[:, 7] > 0
        t1, t2, a = cell(j), cell(j + 1), place(j)
        t = torch.where(use, t1 * (1 - a) + t2 * a, t)
        w = torch.where(use, t2 - t1, w)
    return seg, t, w


def _corners(uv, G):
    """Corner vertices [n, 8], weights [n, 8] and their derivatives with respect to uv [n, 8, 3]."""
    x = (uv + 1) / 2 * (G - 1)
    x0 = torch.floor(x)
    f = x - x0
    idx, w, dw = [], [], []
    for k in range(8):
        bit = [(k >> i) & 1 for i in range(3)]
        c = [(x0[:, i].long() + bit[i]).clamp(0, G - 1) for i in range(3)]
        a = [f[:, i] if bit[i] else 1 - f[:, i] for i in range(3)]
        sg = [(G - 1) / 2 * (1 if b else -1) for b in bit]
        idx.append((c[2] * G + c[1]) * G + c[0])
        w.append(a[0] * a[1] * a[2])
        dw.append(torch.stack([sg[0] * a[1] * a[2], sg[1] * a[0] * a[2], sg[2] * a[0] * a[1]], 1))
    return torch.stack(idx, 1), torch.stack(w, 1), torch.stack(dw, 1)


def _layers(params, H):
    out, at = [], 0
    for fi, fo in ((C, H), (H, H), (H, 1)):
        out.append((params[at:at + fi * fo].double().view(fo, fi), params[at + fi * fo:at + fi * fo + fo].double()))
        at += fi * fo + fo
    return out


def _mlp64(x, L, act, gy=None):
    """softplus(decoder(x)) and, for an upstream gradient, (parameter gradient, dL/dx)."""
    sig = torch.sigmoid
    f = (lambda z: z.clamp(min=0)) if act == "relu" else (lambda z: z * sig(z))
    df = (lambda z: (z > 0).double()) if act == "relu" else (lambda z: sig(z) * (1 + z * (1 - sig(z))))
    z1 = x @ L[0][0].T + L[0][1]
    h1 = f(z1)
    z2 = h1 @ L[1][0].T + L[1][1]
    h2 = f(z2)
    z = (h2 @ L[2][0].T + L[2][1])[:, 0]
    y = torch.nn.functional.softplus(z, beta=BETA, threshold=20)
    if gy is None:
        return y
    dz = (gy * torch.where(z * BETA > 20, torch.ones_like(z), sig(z * BETA)))[:, None]
    d2 = dz @ L[2][0] * df(z2)
    d1 = d2 @ L[1][0] * df(z1)
    parts = [d1.T @ x, d1.sum(0), d2.T @ h1, d2.sum(0), dz.T @ h2, dz.sum(0)]
    return y, torch.cat([p.reshape(-1) for p in parts]), d1 @ L[0][0]


def _exact_projector(case, s):
    sc, G = s["sc"], s["sc"]["G"]
    g = _segments(case, s)
    if case.get("proposal"):
        g["n"], g["cdf"] = _proposal64(s, g)
    flat = s["grid"].permute(0, 2, 3, 4, 1).reshape(-1, C)
    L = _layers(s["params"], sc["H"])
    ends = torch.cumsum(g["n"], 0)
    total, cuts = int(ends[-1]) if len(ends) else 0, [0]
    for q in range(1, max(1, -(-total // (1 << 20)))):
        cuts.append(int(torch.searchsorted(ends, q << 20)))
    cuts = sorted(set(cuts + [len(ends)]))
    o, d = s["o"].double(), s["d"].double()
    proj = torch.zeros(len(o), dtype=torch.float64, device=o.device)

    def chunk(k0, k1):
        seg, t, w = _samples(case, s, g, k0, k1, case["kind"] == "step")
        ray, slot = g["ray"][seg], g["slot"][seg]
        p = o[ray] + d[ray] * t[:, None]
        box = g["mx"][slot] - g["mn"][slot]
        idx, cw, dw = _corners((p - g["mn"][slot]) / box * 2 - 1, G)
        idx = idx + (slot * G ** 3)[:, None]
        x = torch.zeros(len(seg), C, dtype=torch.float64, device=o.device)
        for k in range(8):
            x += flat[idx[:, k]].double() * cw[:, k:k + 1]
        return ray, t, w, box, idx, cw, dw, x

    for k0, k1 in zip(cuts, cuts[1:]):
        ray, t, w, box, idx, cw, dw, x = chunk(k0, k1)
        proj.index_add_(0, ray, _mlp64(x, L, case["act"]) * w)
    if case["kind"] == "view":
        return {"proj": proj}
    gproj = 2 * (proj - s["target"].double()) / len(o)
    gg = torch.zeros(flat.shape, dtype=torch.float64, device=o.device)
    gp = torch.zeros(s["params"].numel(), dtype=torch.float64, device=o.device)
    go, gd = torch.zeros_like(o), torch.zeros_like(d)
    for k0, k1 in zip(cuts, cuts[1:]):
        ray, t, w, box, idx, cw, dw, x = chunk(k0, k1)
        _, dp, dx = _mlp64(x, L, case["act"], gproj[ray] * w)
        gp += dp
        guv = torch.zeros(len(ray), 3, dtype=torch.float64, device=o.device)
        for k in range(8):
            gg.index_add_(0, idx[:, k], dx * cw[:, k:k + 1])
            if case["pose"]:
                guv += dw[:, k] * (flat[idx[:, k]].double() * dx).sum(1, keepdim=True)
        if case["pose"]:
            pos = guv * 2 / box
            go.index_add_(0, ray, pos)
            gd.index_add_(0, ray, pos * t[:, None])
    out = {"proj": proj, "grid": _planes(gg, s["grid"]), "params": gp}
    if case["pose"]:
        out["origin"], out["direction"] = go, gd
    return out


def _planes(flat, grid):
    """[slots * G^3, C] in the grid's [slots, C, G, G, G] indexing."""
    return flat.view(grid.shape[0], *grid.shape[2:], C).permute(0, 4, 1, 2, 3)


def _exact_gather(case, s):
    """At the FP32 local coordinates that the framework is given."""
    G, flat = s["sc"]["G"], s["grid"].permute(0, 2, 3, 4, 1).reshape(-1, C)
    slot, uv, gout = s["slot"], s["uv"], s["gout"]
    S = len(slot)
    feat = torch.zeros(S, C, dtype=torch.float64, device=slot.device)
    guv = torch.zeros(S, 3, dtype=torch.float64, device=slot.device)
    gg = torch.zeros(flat.shape, dtype=torch.float64, device=slot.device)
    for a in range(0, S, 1 << 20):
        r = slice(a, a + (1 << 20))
        idx, cw, dw = _corners(uv[r].double(), G)
        idx = idx + (slot[r] * G ** 3)[:, None]
        go = gout[r].double()
        for k in range(8):
            v = flat[idx[:, k]].double()
            feat[r] += v * cw[:, k:k + 1]
            guv[r] += dw[:, k] * (v * go).sum(1, keepdim=True)
            gg.index_add_(0, idx[:, k], go * cw[:, k:k + 1])
    return {"feat": feat, "grid": _planes(gg, s["grid"]), "uv": guv}


def _active_at(t, q, dev):
    """The active node that holds the points q [M, 3] (float32): from the root, through inactive nodes, the first
    child whose closed box holds the point; -1 if there is none."""
    pmin, pmax = torch.from_numpy(t["pmin"]).to(dev), torch.from_numpy(t["pmax"]).to(dev)
    act = torch.from_numpy(t["active"]).to(dev) > 0
    n = torch.zeros(len(q), dtype=torch.long, device=dev)
    res = torch.full_like(n, -1)
    open_ = torch.ones(len(q), dtype=torch.bool, device=dev)
    for level in range(t["depth"] + 1):
        done = open_ & act[n]
        res[done] = n[done]
        open_ &= ~done
        if level == t["depth"]:
            break
        nxt = torch.full_like(n, -1)
        for c in range(7, -1, -1):
            ch = 8 * n + 1 + c
            nxt = torch.where(((pmin[ch] <= q) & (pmax[ch] >= q)).all(1), ch, nxt)
        open_ &= nxt >= 0
        n = torch.where(open_, nxt, torch.zeros_like(n))
    return res


def _exact_reg(case, s, loss_tv=1e-4, loss_edge=1e-3):
    t, grid = s["tree"], s["grid"].double()
    dev, G, A = grid.device, s["sc"]["G"], len(t["ids"])
    gg, loss = torch.zeros_like(grid), 0.0
    for ax in (2, 3, 4):
        diff = grid.narrow(ax, 1, G - 1) - grid.narrow(ax, 0, G - 1)
        scale = loss_tv * C / (A * C * G * G * (G - 1))
        loss = loss + diff.abs().sum() * scale
        sg = torch.sign(diff) * scale
        gg.narrow(ax, 1, G - 1).add_(sg)
        gg.narrow(ax, 0, G - 1).sub_(sg)
        del diff, sg
    ids, prefix = torch.from_numpy(t["ids"]).to(dev), torch.from_numpy(t["prefix"]).to(dev)
    pmin, pmax = torch.from_numpy(t["pmin"]).to(dev), torch.from_numpy(t["pmax"]).to(dev)
    sid = torch.arange(G * G, device=dev)
    lane = torch.stack([(sid % G).float() / (float(G) - 1.0), (sid // G).float() / (float(G) - 1.0)], 1)
    rows = []  # [A, 6, G^2]: neighbour, point
    for side in range(3):
        for front in range(2):
            local = torch.zeros(G * G, 3, device=dev)
            local[:, side] = float(front)
            local[:, (side + 1) % 3], local[:, (side + 2) % 3] = lane[:, 0], lane[:, 1]
            mn, mx = pmin[ids][:, None], pmax[ids][:, None]
            p = (local[None] * (mx - mn) + mn).reshape(-1, 3)
            q = p.clone()
            q[:, side] += 0.001 if front else -0.001
            rows.append((_active_at(t, q, dev).view(A, 1, -1), p.view(A, 1, G * G, 3)))
    other, p = torch.cat([r[0] for r in rows], 1).reshape(-1), torch.cat([r[1] for r in rows], 1).reshape(-1, 3)
    node = ids[:, None].expand(A, 6 * G * G).reshape(-1)
    pair = (other >= 0) & (other != node)
    node, other, p = node[pair], other[pair], p[pair].double()
    P = len(node)
    flat, fg = grid.permute(0, 2, 3, 4, 1).reshape(-1, C), torch.zeros(A * G ** 3, C, dtype=torch.float64, device=dev)
    for a in range(0, P, 1 << 20):
        r = slice(a, min(P, a + (1 << 20)))
        f, keep = [], []
        for n in (node[r], other[r]):
            mn, mx = pmin[n].double(), pmax[n].double()
            idx, cw, _ = _corners((p[r] - mn) / (mx - mn) * 2 - 1, G)
            idx = idx + (prefix[n] * G ** 3)[:, None]
            f.append(sum(flat[idx[:, k]] * cw[:, k:k + 1] for k in range(8)))
            keep.append((idx, cw))
        k = torch.arange(r.start, r.stop, device=dev)
        fac = _unit24(_mix64(torch.tensor(s["seed"], device=dev) ^ (k * _GOLD)))[:, None]
        diff = f[0] - f[1]
        loss = loss + (diff.abs() * fac).sum() * loss_edge / P
        g = torch.sign(diff) * fac * loss_edge / P
        for (idx, cw), sg in zip(keep, (1.0, -1.0)):
            for c in range(8):
                fg.index_add_(0, idx[:, c], g * cw[:, c:c + 1] * sg)
    return {"loss": loss.reshape(1), "grid": gg + _planes(fg, grid)}


def exact(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    if kind in ("view", "step"):
        return _exact_projector(case, s)
    if kind == "gather":
        return _exact_gather(case, s)
    if kind == "mlp":
        L = _layers(s["params"], case["hidden"])
        y, gp, gx = [], 0.0, []
        for a in range(0, case["rows"], 1 << 20):
            r = slice(a, a + (1 << 20))
            o = _mlp64(s["x"][r].double(), L, case["act"], s["gy"][r, 0].double())
            y.append(o[0][:, None])
            gp = gp + o[1]
            gx.append(o[2])
        return {"y": torch.cat(y), "params": gp, "x": torch.cat(gx)}
    if kind == "reg":
        return _exact_reg(case, s)
    out = {}
    for n, lr, names in (("grid", 1e-2, ("grid", "m", "v")), ("params", 1e-3, ("params", "pm", "pv"))):
        p, g, m, v = (t.double() for t in s[n])
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - lr / (1 - 0.9 ** s["step"]) * m / (v.sqrt() / math.sqrt(1 - 0.999 ** s["step"]) + 1e-8)
        out.update(zip(names, (p, m, v)))
    return {"grid": out["grid"], "m": out["m"], "v": out["v"], "bf16": None, "params": out["params"],
            "pm": out["pm"], "pv": out["pv"]}
