"""The calls whose speed this framework is judged by, as a user's program makes
them: the drop-in ray ops (`nsvf_amd.clib`), the differentiable gather and
field MLP and a whole training step (`nsvf_amd.train`), whole views
(`nsvf_amd.render`) and pruning (`nsvf_amd.voxels`).

A case is a dict of plain values; `prepare` makes what a program holds before
the call (on the GPU, from a seed), `run` makes the call, `work` says what the
call cannot do without and `exact` gives its float outputs in 64 bits where
they have such a value.

Scenes are the synthetic ones of `nsvf_amd.scene`: the spherical shell (32^3
grid: 6,568 voxels) and the value-noise cloud on a 128^3 grid (100,000 voxels
in the headline view).  Their voxel grids are fixed; embeddings, MLP weights,
cameras, pixels and gradients come from the seed.
"""
from __future__ import annotations

import functools
import math
from dataclasses import replace

import numpy as np
import torch

from nsvf_amd import clib, geometry, voxels
from nsvf_amd import scene as S
from nsvf_amd import train
from nsvf_amd.render import DeviceScene, Renderer

DEV = "cuda:0"


def listed():
    return [
        # a training batch's rays against the octree through the drop-in op:
        # 4 views x 2,048 random pixels of the shell, unrelated neighbours
        dict(name="svo_batch", kind="svo", grid="shell", res=32, rays=8192, order="random"),
        # a 401 x 399 image against the octree of the 100k-voxel cloud, as the
        # reference's renderer calls the op
        dict(name="svo_view", kind="svo", grid="noise", voxels=100_000, rays=401 * 399,
             order="image"),
        # the encoder's other intersection (no octree): brute force over the
        # shell's voxels for a training batch
        dict(name="aabb_batch", kind="aabb", grid="shell", res=32, rays=8192, order="random"),
        # inverse-CDF samples of an image's hit rows (evaluation: no noise)
        dict(name="icdf_view", kind="icdf", rows=65_537, bins=60, noise=False),
        # the trilinear gather of a training step and its backward, scene of
        # 100k voxels
        dict(name="gather_train", kind="gather", grid="noise", voxels=100_000, samples=800_003),
        # the field MLP forward and backward in the trainer's default FP32: a
        # handful of rays, where launches count
        dict(name="mlp_fp32_small", kind="mlp", precision="fp32", samples=4093),
        # ... and the samples of a 20k-ray batch
        dict(name="mlp_fp32_large", kind="mlp", precision="fp32", samples=1_000_003),
        # a whole training step on the shell, 4 views x 2,048 random pixels,
        # with the split-BF16 MLP (whole steps are listed in this precision
        # only: a step's gradients pass the ReLU kinks of every sample, where
        # two FP32 roundings may take different sides)
        dict(name="train_step", kind="step", res=32, rays_per_view=2048),
        # a preview-sized view at the renderer's default precision
        dict(name="view_small", kind="view", grid="shell", res=32, height=200, width=136,
             precision="bf16", fine=True),
        # a single-pass view in the reference's own precision
        dict(name="view_fp32", kind="view", grid="noise", voxels=100_000, height=400, width=400,
             precision="fp32", fine=False),
        # the headline: an 800 x 800 view at the served precision, coarse and
        # fine pass
        dict(name="view_800", kind="view", grid="noise", voxels=100_000, height=800, width=800,
             precision="bf16x3", fine=True),
        # pruning scores of every voxel of the shell over its 16^3 lattice
        dict(name="prune", kind="prune", grid="shell", res=32, precision="fp32"),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, most=100_000):
    """A shell of 16^3 to 40^3 cells or a noise cloud of 10k voxels and more."""
    if rng.random() < 0.5:
        return dict(grid="shell", res=rng.randint(16, 40))
    return dict(grid="noise", voxels=_log(rng, 10_000, most))


def draw(rng):
    kind = rng.choice(["svo", "aabb", "icdf", "gather", "mlp", "step", "view", "prune"])
    if kind == "svo":
        return dict(kind=kind, **_grid(rng), rays=_log(rng, 500, 160_000),
                    order=rng.choice(["random", "image"]))
    if kind == "aabb":
        return dict(kind=kind, grid="shell", res=rng.randint(16, 36), rays=_log(rng, 300, 10_000),
                    order=rng.choice(["random", "image"]))
    if kind == "icdf":
        return dict(kind=kind, rows=_log(rng, 300, 66_000), bins=rng.randint(20, 60),
                    noise=rng.random() < 0.5)
    if kind == "gather":
        return dict(kind=kind, **_grid(rng), samples=_log(rng, 1000, 800_000))
    if kind == "mlp":
        return dict(kind=kind, precision=rng.choice(["fp32", "bf16x3"]),
                    samples=_log(rng, 500, 1_000_000))
    if kind == "step":
        return dict(kind=kind, res=rng.randint(20, 36), rays_per_view=_log(rng, 100, 3000))
    if kind == "view":
        precision = rng.choice(["bf16", "bf16x3", "fp32"])
        most = 400 if precision == "fp32" else 640
        return dict(kind=kind, **_grid(rng), height=_log(rng, 40, most), width=_log(rng, 40, most),
                    precision=precision, fine=precision != "fp32")
    return dict(kind=kind, grid="shell", res=rng.randint(16, 32),
                precision=rng.choice(["fp32", "bf16x3"]))


# ---------------------------------------------------------------------------
# What a program holds before the call


@functools.lru_cache(maxsize=16)
def _voxel_grid(grid, size):
    """A scene's voxels, corner keys and corner ids (made once per size)."""
    if grid == "shell":
        return S.shell_scene(res=size, embed_dim=4, hidden=16, layers=1)
    return S.noise_scene(res=128, num_voxels=size, embed_dim=4, hidden=16, layers=1)


def _scene(case, seed):
    """The case's voxel grid with seeded 32-d embeddings and 3 x 128 MLP."""
    base = _voxel_grid(case.get("grid", "shell"), case["voxels"] if "voxels" in case else case["res"])
    rng = np.random.default_rng([5, seed])
    values = (rng.standard_normal((base.num_keys, 32), np.float32) * np.float32(0.1))
    return replace(base, embed_dim=32, values=values, mlp=S.make_mlp(32, 128, 3, [6, seed]))


def _shifted(scene):
    """Voxel centres with the gather's x-shift (encoder.py:383)."""
    pts = torch.from_numpy(scene.points.copy())
    pts[:, 0] += torch.tensor(np.float32(scene.voxel_size)) / 10
    return pts.to(DEV)


def _image_rays(height, width, seed):
    cam = S.sphere_camera(2.5, [7, seed])
    rs, rd = S.camera_rays(width, height, cam, focal=1.2 * max(width, height))
    return torch.from_numpy(rs).to(DEV), torch.from_numpy(rd).to(DEV)


def _batch_rays(rays, seed, views=4, res=256):
    """Random pixels of several views, view after view, as training draws them."""
    rng = np.random.default_rng([8, seed])
    starts, dirs = [], []
    for v in range(views):
        n = rays // views + (v < rays % views)
        rs, rd = S.camera_rays(res, res, S.sphere_camera(2.5, [9, seed, v]))
        pick = rng.integers(0, res * res, n)
        starts.append(rs[pick])
        dirs.append(rd[pick])
    return (torch.from_numpy(np.concatenate(starts)).to(DEV),
            torch.from_numpy(np.concatenate(dirs)).to(DEV))


def _op_rays(case, seed):
    n = case["rays"]
    if case["order"] == "random":
        return _batch_rays(n, seed)
    w = max(1, int(round(math.sqrt(n))))
    rs, rd = _image_rays(-(-n // w), w, seed)
    return rs[:n].contiguous(), rd[:n].contiguous()


def _generator(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed(1_000_003 * salt + seed)
    return g


def _hit_rows(rows, bins, seed, vs=2.0 ** -6):
    """Sorted hit rows as the encoder hands them to the sampler
    (encoder.py:518-535): crossings of up to a voxel diagonal, gaps now and
    then, a few rows full, padded with -1 and depth 10,000.  The last row is
    the scene's longest crossing, the same in every image: it sets the
    outputs' width."""
    g = _generator(seed, 11)
    rand = lambda *s: torch.rand(*s, generator=g, device=DEV)
    # most rays cross a dozen voxels, a few fill every slot
    count = (1 - torch.log1p(-rand(rows) * 0.999) * bins / 4).floor().clamp_(1, bins)
    count[-1] = bins
    pad = torch.arange(bins, device=DEV)[None] >= count[:, None]
    length = (rand(rows, bins) * 1.7 + 0.01) * vs
    longest = 0.9 * bins * vs
    length *= (0.96 * longest / length.masked_fill(pad, 0.0).sum(1, keepdim=True)).clamp(max=1.0)
    length[-1] = longest / bins
    gap = torch.where(rand(rows, bins) < 0.15, rand(rows, bins) * 8 * vs, 0.0)
    gap[-1] = 0.0
    hi = 1.5 + torch.cumsum(length + gap, 1)
    lo = hi - length
    idx = torch.randint(0, 100_000, (rows, bins), generator=g, device=DEV, dtype=torch.int32)
    idx = idx.masked_fill(pad, -1)
    lo, hi = lo.masked_fill(pad, clib.MAX_DEPTH), hi.masked_fill(pad, clib.MAX_DEPTH)
    dists = (hi - lo).masked_fill(pad, 0.0)
    total = dists.sum(-1)
    return idx, lo, hi, dists / total[:, None], total / (vs / 8)


def _gather_inputs(case, scene, seed):
    """A ray-ordered sample stream: rays crossing about 8 voxels with a few
    samples in each, two unused slots after every ray."""
    M, N = case["samples"], scene.num_voxels
    g = _generator(seed, 12)
    per = 8 * 6 + 2
    i = torch.arange(M, device=DEV)
    ray, slot = i // per, i % per
    first = torch.randint(0, N, (M // per + 1,), generator=g, device=DEV)
    s_idx = ((first[ray] + slot // 6) % N).int()
    s_idx = torch.where(slot >= 48, -1, s_idx).int()
    cen = _shifted(scene)
    u = torch.rand(M, 3, generator=g, device=DEV) - 0.5
    xyz = cen[s_idx.clamp(min=0).long()] + u * scene.voxel_size
    grad = torch.randn(M, 32, generator=g, device=DEV) * 1e-3
    return s_idx, xyz, cen, grad


def _mlp_double(x, params, kinks=False):
    """The field MLP in 64 bits: [M, 32] -> [M, 4] (sigma, r, g, b); with
    kinks also each sample's smallest hidden |pre-activation|."""
    h, near = x, None
    for k in range(0, len(params) - 2, 2):
        z = h @ params[k].T + params[k + 1]
        if kinks:
            m = z.abs().amin(1)
            near = m if near is None else torch.minimum(near, m)
        h = torch.relu(z)
    z = h @ params[-2].T + params[-1]
    out = torch.cat([z[:, :1], torch.sigmoid(z[:, 1:])], 1)
    return (out, near) if kinks else out


_CHUNK = 1 << 18   # samples per piece of the 64-bit MLP


def _mlp_inputs(case, seed):
    g = _generator(seed, 13)
    M = case["samples"]
    mlp = S.make_mlp(32, 128, 3, [6, seed])
    params = []
    for w, b in zip(mlp.weights, mlp.biases):
        params += [torch.from_numpy(w).to(DEV), torch.from_numpy(b).to(DEV)]
    emb = torch.randn(M, 32, generator=g, device=DEV) * 0.1
    # the image loss reaches a sample through its compositing weight, which
    # falls over orders of magnitude along a ray; samples outside every ray
    # have none
    scale = 10.0 ** (-4 * torch.rand(M, 1, generator=g, device=DEV)) / M
    dout = torch.randn(M, 4, generator=g, device=DEV) * scale
    dout[torch.rand(M, generator=g, device=DEV) < 0.05] = 0
    # a sample within the arithmetic's rounding of a ReLU kink has two
    # gradients, one per side: it gets none
    margin = 2e-6 if case["precision"] == "fp32" else 1e-4
    p64 = [p.double() for p in params]
    for a in range(0, M, _CHUNK):
        near = _mlp_double(emb[a:a + _CHUNK].double(), p64, kinks=True)[1]
        dout[a:a + _CHUNK][near < margin] = 0
    return emb, params, dout


def prepare(case, seed):
    kind = case["kind"]
    if kind == "svo":
        scene = _scene(case, seed)
        cen, ch = geometry.build_easy_octree(torch.from_numpy(scene.points),
                                             torch.tensor(np.float32(scene.voxel_size)) / 2)
        rs, rd = _op_rays(case, seed)
        return dict(kind=kind, scene=scene, nodes=cen.to(DEV)[None], children=ch.to(DEV)[None],
                    rs=rs[None], rd=rd[None])
    if kind == "aabb":
        scene = _scene(case, seed)
        rs, rd = _op_rays(case, seed)
        return dict(kind=kind, scene=scene, points=_shifted(scene)[None], rs=rs[None], rd=rd[None])
    if kind == "icdf":
        rows = _hit_rows(case["rows"], case["bins"], seed)
        noise = steps = None
        if case["noise"]:
            steps = int(rows[4].ceil().max().item()) + case["bins"]
            noise = torch.rand(case["rows"], steps, generator=_generator(seed, 14),
                               device=DEV).clamp_(0.001, 0.999)
        return dict(kind=kind, rows=rows, noise=noise, steps=steps)
    if kind == "gather":
        scene = _scene(case, seed)
        s_idx, xyz, cen, grad = _gather_inputs(case, scene, seed)
        feats = torch.from_numpy(scene.feats.astype(np.int32)).to(DEV)
        values = torch.from_numpy(scene.values).to(DEV).requires_grad_()
        return dict(kind=kind, values=values, s_idx=s_idx, xyz=xyz, centers=cen, feats=feats,
                    vs=scene.voxel_size, grad=grad,
                    plan=train.gather_backward_plan(feats, scene.num_keys))
    if kind == "mlp":
        emb, params, dout = _mlp_inputs(case, seed)
        fn = train.FieldMLP if case["precision"] == "fp32" else train.FieldMLPx3
        leaves = [t.requires_grad_() for t in (emb, *params)]
        return dict(kind=kind, fn=fn, leaves=leaves, dout=dout)
    if kind == "step":
        scene = _scene(case, seed)
        n = 4 * case["rays_per_view"]
        rs, rd = _batch_rays(n, seed)
        target = torch.rand(n, 3, generator=_generator(seed, 15), device=DEV)
        return dict(kind=kind, scene=DeviceScene(scene, DEV),
                    field=train.TrainableField(scene, DEV, mlp="hip_x3"),
                    renderer=train.TrainRenderer(DEV), rs=rs, rd=rd, target=target, noise=seed)
    if kind == "view":
        rs, rd = _image_rays(case["height"], case["width"], seed)
        return dict(kind=kind, scene=DeviceScene(_scene(case, seed), DEV), rs=rs, rd=rd,
                    width=case["width"],
                    renderer=Renderer(DEV, precision=case["precision"], hierarchical=case["fine"]))
    if kind == "prune":
        return dict(kind=kind, scene=DeviceScene(_scene(case, seed), DEV),
                    precision=case["precision"])
    raise ValueError(f"kind {kind!r}")


# ---------------------------------------------------------------------------
# The call


def run(state):
    kind = state["kind"]
    if kind == "svo":
        sc = state["scene"]
        return clib.svo_ray_intersect(sc.voxel_size, sc.max_hits, state["nodes"],
                                      state["children"], state["rs"], state["rd"])
    if kind == "aabb":
        sc = state["scene"]
        return clib.aabb_ray_intersect(sc.voxel_size, sc.max_hits, state["points"], state["rs"],
                                       state["rd"])
    if kind == "icdf":
        if state["noise"] is None:
            return clib.inverse_cdf_sampling(*state["rows"], -1, True)
        return clib.inverse_cdf_sampling_rows(*state["rows"], noise=state["noise"],
                                              max_steps=state["steps"])[:3]
    if kind == "gather":
        emb = train.trilinear_gather(state["values"], state["s_idx"], state["xyz"],
                                     state["centers"], state["feats"], state["vs"], state["plan"])
        (grad,) = torch.autograd.grad(emb, [state["values"]], state["grad"])
        return dict(emb=emb, grad_values=grad)
    if kind == "mlp":
        out = state["fn"].apply(*state["leaves"])
        return dict(out=out, grads=torch.autograd.grad(out, state["leaves"], state["dout"]))
    if kind == "step":
        field = state["field"]
        field.zero_grad(set_to_none=True)
        rgb, depth, missed = state["renderer"].forward(state["scene"], field, state["rs"],
                                                       state["rd"], seed=state["noise"])
        train.mse_loss(rgb, state["target"]).backward()
        return dict(rgb=rgb, depth=depth, missed=missed,
                    grads=[p.grad for p in field.parameters()])
    if kind == "view":
        return state["renderer"].render(state["scene"], state["rs"], state["rd"],
                                        width=state["width"])
    return voxels.prune_scores(state["scene"], state["precision"])


# ---------------------------------------------------------------------------
# What a call cannot do without

MLP_FLOPS = 2 * (32 * 128 + 2 * 128 * 128 + 128 * 4)   # per sample
MLP_BYTES = 4 * (32 * 128 + 2 * 128 * 128 + 128 * 4 + 3 * 128 + 4)


def work(case):
    kind = case["kind"]
    grid = None
    if "grid" in case or kind == "step":
        grid = _voxel_grid(case.get("grid", "shell"),
                           case["voxels"] if "voxels" in case else case["res"])
    if kind in ("svo", "aabb"):
        # rays in, 60 slots of (id, entry, exit) per ray out, the scene once;
        # a slab test (about 20 operations) per returned hit and box passed
        scene = grid.num_voxels * (12 if kind == "aabb" else 2.2 * 48)
        return dict(bytes=case["rays"] * (24 + 60 * 12) + scene, flops=case["rays"] * 60 * 20)
    if kind == "icdf":
        # bins in, out padded rows of the longest row's steps (7.2 per bin)
        # and one sample more per bin
        slots = case["bins"] * 8.2
        return dict(bytes=case["rows"] * (case["bins"] * 16 + 4 + slots * 12
                                          + (slots * 4 if case["noise"] else 0)),
                    flops=case["rows"] * slots * 8)
    if kind == "gather":
        M, K, N = case["samples"], grid.num_keys, grid.num_voxels
        return dict(bytes=M * (16 + 2 * 128) + N * 44 + 2 * K * 128, flops=M * 8 * 32 * 4)
    if kind == "mlp":
        M = case["samples"]
        return dict(bytes=M * (128 + 16 + 16 + 128) + 2 * MLP_BYTES, flops=M * 3 * MLP_FLOPS)
    if kind == "step":
        # about 35 samples per ray of the shell's image
        M, K, N = 35 * 4 * case["rays_per_view"], grid.num_keys, grid.num_voxels
        return dict(bytes=M * 64 + 2 * K * 128 + N * 44 + 2 * MLP_BYTES, flops=M * 3 * MLP_FLOPS)
    if kind == "view":
        # about 47 coarse samples per pixel, 60 more to evaluate in a fine pass
        R = case["height"] * case["width"]
        M = R * (107 if case["fine"] else 47)
        return dict(bytes=R * (24 + 20) + grid.num_keys * 128 + grid.num_voxels * 44,
                    flops=M * MLP_FLOPS)
    return dict(bytes=grid.num_keys * 128 + grid.num_voxels * 48,
                flops=grid.num_voxels * 4096 * MLP_FLOPS)


# ---------------------------------------------------------------------------
# The float outputs in 64 bits.  The ray ops, views and steps have none: their
# float outputs are placed by whole-number decisions (which box is hit, which
# bin a step falls in) that 64-bit arithmetic takes differently now and then.


def exact(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        emb, params, dout = _mlp_inputs(case, seed)
        p64 = [p.double().requires_grad_() for p in params]
        outs, dembs, total = [], [], None
        for a in range(0, case["samples"], _CHUNK):
            x = emb[a:a + _CHUNK].double().requires_grad_()
            out = _mlp_double(x, p64)
            grads = torch.autograd.grad(out, [x, *p64], dout[a:a + _CHUNK].double())
            outs.append(out.detach())
            dembs.append(grads[0])
            total = list(grads[1:]) if total is None else [s + t for s, t in zip(total, grads[1:])]
        return dict(out=torch.cat(outs), grads=(torch.cat(dembs), *total))
    if kind == "gather":
        scene = _scene(case, seed)
        s_idx, xyz, cen, grad = _gather_inputs(case, scene, seed)
        feats = torch.from_numpy(scene.feats).to(DEV)
        values = torch.from_numpy(scene.values).to(DEV).double()
        used = s_idx >= 0
        v = s_idx.clamp(min=0).long()
        p = (xyz.double() - cen[v].double()) / scene.voxel_size + 0.5
        emb = torch.zeros(case["samples"], 32, dtype=torch.float64, device=DEV)
        out = torch.zeros_like(values)
        for c in range(8):
            w = torch.ones_like(p[:, 0])
            for a, bit in enumerate((4, 2, 1)):
                w = w * (p[:, a] if c & bit else 1 - p[:, a])
            w = torch.where(used, w, 0.0)[:, None]
            emb += w * values[feats[v, c]]
            out.index_add_(0, feats[v, c], w * grad.double())
        return dict(emb=emb, grad_values=out)
    if kind == "prune":
        scene = _scene(case, seed)
        cen = _shifted(scene)
        feats = torch.from_numpy(scene.feats).to(DEV)
        values = torch.from_numpy(scene.values).to(DEV).double()
        params = []
        for w, b in zip(scene.mlp.weights, scene.mlp.biases):
            params += [torch.from_numpy(w).to(DEV).double(), torch.from_numpy(b).to(DEV).double()]
        # the lattice points as 32-bit positions (encoder.py:620-646), then
        # their corner weights and field in 64 bits
        i = torch.arange(16, dtype=torch.float32, device=DEV)
        off = (2 * i + 1 - 16) / 15.0
        ox, oy, oz = torch.meshgrid(off, off, off, indexing="ij")
        half = torch.tensor(np.float32(scene.voxel_size) * np.float32(0.5), device=DEV)
        offs = torch.stack([ox.reshape(-1), oy.reshape(-1), oz.reshape(-1)], 1) * half
        best = []
        for v0 in range(0, scene.num_voxels, 64):
            c = cen[v0:v0 + 64]
            p = ((c[:, None] + offs[None]).double() - c[:, None].double()) / scene.voxel_size + 0.5
            q = 1 - p
            w = torch.stack([(p[..., 0] if k & 4 else q[..., 0]) * (p[..., 1] if k & 2 else q[..., 1])
                             * (p[..., 2] if k & 1 else q[..., 2]) for k in range(8)], -1)
            emb = w @ values[feats[v0:v0 + 64]]
            sigma = _mlp_double(emb.reshape(-1, 32), params)[:, 0]
            best.append(sigma.view(c.shape[0], -1).clamp(min=0).amax(1))
        return torch.cat(best)
    return None
