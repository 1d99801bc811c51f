"""The work that a user of this package has it do: inference and training of Flash3D models on batches of LiDAR sweeps,
and the operators they are made of, called on their own (bucketing, one block, pooling, attention).

    listed()               the cases by name
    draw(rng)              another case of the same ranges
    prepare(case, seed)    inputs, model and buffers a program has in hand before the call, on the GPU
    run(state)             one pass through the public entry points; returns its outputs
    work(case)             bytes and operations of one pass that no implementation can do without
    tolerance(case)        how far two correct implementations at this precision may be apart

Sizes follow the benchmark workloads and tests of this repository: buckets of 512 rows, 32-wide heads, hidden width
4 C, five levels of 32 to 512 channels, LiDAR sweeps of 120,000 / 250,000 points, clouds of 32,768 points."""
import math
from functools import partial

import torch
from torch import nn

from flash3dtransformer_amd import layers as L
from flash3dtransformer_amd.lib import pshattn
from flash3dtransformer_amd.psh import psh_main
from flash3dtransformer_amd.psh.bucket_scope import SwinPlan, swinable_alignment

DEV = "cuda:0"
BUCKET = 512


def listed():
    return [
        # one small cloud put into hash buckets: the smallest call, bound by launches and the host
        dict(name="bucket_1x32k", kind="bucket", clouds=1, points=32768, ragged=False, hash=1),
        # the bucketing of a whole batch of large clouds: a data pipeline that prepares many sweeps at once
        dict(name="bucket_64x262k", kind="bucket", clouds=64, points=262144, ragged=False, hash=2),
        # the first encoder stage on four sweeps, inference: bucketing, coordinate embedding, one block of 256 channels
        dict(name="stage_4x120k", kind="stage", clouds=4, points=120000, ragged=False, channels=256, scope=1, hash=2),
        # one block on stored features, inference, ragged batch: any block of a model but the first
        dict(name="block_3x97k", kind="block", clouds=3, points=97531, ragged=True, channels=256, scope=1),
        # a five-level model on one small cloud, inference: a detector that answers one sweep at a time
        dict(name="model_1x20k", kind="model", shape="plain", clouds=1, points=20000, ragged=False, levels=5, features=0,
             train=False),
        # the same model on four full sweeps: offline inference
        dict(name="model_4x250k", kind="model", shape="plain", clouds=4, points=250000, ragged=False, levels=5,
             features=0, train=False),
        # the deeper model shape (scopes of 8 buckets, two blocks a side, BatchNorm + GELU around pooling), inference
        dict(name="wide_scope_model_4x120k", kind="model", shape="wide_scope", clouds=4, points=120000, ragged=False,
             levels=5, features=0, train=False),
        # segmentation of a ragged batch: intensity as a point feature, results back in the order the points came in
        dict(name="features_3x83k", kind="model", shape="plain", clouds=3, points=83333, ragged=True, levels=4,
             features=4, train=False),
        # a training step (forward and backward, fp32 master weights) of the five-level model
        dict(name="train_4x120k", kind="model", shape="plain", clouds=4, points=120000, ragged=False, levels=5,
             features=0, train=True),
        # a training step of the deeper shape on a smaller ragged batch, batch statistics in its BatchNorm layers
        dict(name="train_wide_scope_2x60k", kind="model", shape="wide_scope", clouds=2, points=60001, ragged=True,
             levels=5, features=0, train=True),
        # pooling and unpooling on their own, forward and backward: 2 x 2 x 2 reduction of 128 channels
        dict(name="pool_262k", kind="pool", clouds=1, points=262144, ragged=False, channels=128, subbuck=8, op="mean"),
        # the attention operator on partly filled buckets, forward and backward
        dict(name="attention_2x64k_masked", kind="attention", rows=131072, heads=8, head_dim=32, scope=1, masked=True),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    # clouds of fewer than about 9,000 points have fewer than the 32 hash buckets that the bucketing takes
    kind = rng.choice(["bucket", "stage", "block", "model", "model", "model", "model", "pool", "attention"])
    ragged = rng.random() < 0.5
    if kind == "bucket":
        clouds = spread(1, 64)
        return dict(kind=kind, clouds=clouds, points=spread(11000, 262144), ragged=ragged and clouds > 1,
                    hash=rng.choice([1, 2]))
    clouds = rng.choice([1, 2, 3, 4])
    if kind == "stage":
        return dict(kind=kind, clouds=clouds, points=spread(11000, 120000), ragged=ragged,
                    channels=rng.choice([32, 64, 128, 256]), scope=1, hash=rng.choice([1, 2]))
    if kind == "block":
        channels = rng.choice([32, 64, 128, 256, 512])
        return dict(kind=kind, clouds=clouds, points=spread(2000, 60000 if channels == 512 else 120000), ragged=ragged,
                    channels=channels, scope=rng.choice([1, 1, 8]))
    if kind == "pool":
        channels = rng.choice([32, 64, 128, 256])
        return dict(kind=kind, clouds=clouds, points=spread(11000, min(262144, (29 << 20) // (clouds * channels))),
                    ragged=ragged, channels=channels, subbuck=rng.choice([2, 2, 4, 8]), op=rng.choice(["mean", "max"]))
    if kind == "attention":
        scope = rng.choice([1, 1, 2, 4, 8])
        heads, head_dim = rng.choice([(2, 16), (4, 16), (2, 32), (4, 32), (8, 32), (2, 64), (4, 64)])
        return dict(kind=kind, rows=BUCKET * scope * max(1, spread(4000, 131072) // (BUCKET * scope)), heads=heads,
                    head_dim=head_dim, scope=scope, masked=rng.random() < 0.5)
    shape, train = rng.choice(["plain", "plain", "wide_scope"]), rng.random() < 0.5
    top = {("plain", False): 250000, ("plain", True): 120000, ("wide_scope", False): 120000, ("wide_scope", True): 30000}
    return dict(kind=kind, shape=shape, clouds=clouds, points=spread(11000, top[shape, train]), ragged=ragged,
                levels=rng.choice([3, 4, 5]), features=rng.choice([0, 0, 4]), train=train)


# ------------------------------------------------------------------------------------------------ sizes

def _sizes(case):
    """points of every cloud; those of a ragged batch are spread around the stated size"""
    n, b = case["points"], case["clouds"]
    if not case["ragged"]:
        return [n] * b
    return [int(n * (0.7 + 0.6 * ((0.618 * i + 0.4) % 1.0))) + 3 * i for i in range(b)]


def _up(n, m):
    return -(-n // m) * m


def _channels(case):
    return [32 << i for i in range(case["levels"])]


def _model_shape(case):
    """(scope, blocks per side and level)"""
    return (1, 1) if case["shape"] == "plain" else (8, 2)


# ------------------------------------------------------------------------------------------------ inputs

def _sweep(n, g):
    """n points of a spinning LiDAR: 64 elevation rings from -25 to +2 degrees, rays against a ground plane 1.7 m below
    and 30 boxes, ranges of 2 to 80 m, thinned by 1 / r^2; points in ring order, with an intensity in [0, 1)"""
    rays = 3 * n + 4096
    u = lambda *shape: torch.rand(*shape, device=DEV, generator=g)
    ring = torch.arange(rays, device=DEV) * 64 // rays
    e = torch.deg2rad(-25.0 + 27.0 / 63.0 * ring) + math.radians(0.05) * torch.randn(rays, device=DEV, generator=g)
    a = u(rays) * (2.0 * math.pi)
    d = torch.stack([torch.cos(e) * torch.cos(a), torch.cos(e) * torch.sin(a), torch.sin(e)], dim=1)
    inv = 1.0 / torch.where(d.abs() < 1e-9, torch.full_like(d, 1e-9), d)
    t = torch.where(d[:, 2] < 0, -1.7 * inv[:, 2], torch.full_like(a, math.inf))
    c, s = (u(30, 2) - 0.5) * 120.0, 1.0 + 5.0 * u(30, 3)
    lo = torch.cat([c - s[:, :2] / 2, torch.full((30, 1), -1.7, device=DEV)], dim=1)
    hi = torch.cat([c + s[:, :2] / 2, s[:, 2:] - 1.7], dim=1)
    for k in range(0, 30, 10):
        p, q = lo[k:k + 10, None] * inv, hi[k:k + 10, None] * inv
        near, far = torch.minimum(p, q).amax(-1), torch.maximum(p, q).amin(-1)
        hit = torch.where((far >= near) & (near > 0), near, torch.full_like(near, math.inf))
        t = torch.minimum(t, hit.amin(0))
    kept = (t >= 2.0) & (t <= 80.0)
    # weighted sampling without replacement: the n largest of log(u) / w, w = 1 / r^2
    key = torch.where(kept, torch.log(u(rays).clamp_min(1e-12)) * t.clamp(2.0, 80.0) ** 2, torch.full_like(t, -math.inf))
    idx = torch.topk(key, n, sorted=False).indices.sort().values
    return torch.cat([d[idx] * t[idx, None], u(n, 1)], dim=1)


def _batch(case, g):
    """(coords [N, 3] fp16, seps [B] uint32, points [N, 4] fp32)"""
    sizes = _sizes(case)
    pts = torch.cat([_sweep(n, g) for n in sizes])
    seps = torch.tensor(sizes, dtype=torch.int64).cumsum(0).to(torch.int32).to(DEV).view(torch.uint32)
    return pts[:, :3].to(torch.float16).contiguous(), seps, pts


def _trained_(module, g):
    """affine and statistics parameters as they are after some training, not at their initial ones and zeros"""
    with torch.no_grad():
        for m in module.modules():
            if isinstance(m, nn.BatchNorm1d):
                m.running_mean.copy_(torch.randn(m.num_features, generator=g) * 0.1)
                m.running_var.copy_(torch.rand(m.num_features, generator=g) + 0.5)
            if isinstance(m, (L.LayerNorm, nn.BatchNorm1d)):
                m.weight.copy_(torch.rand(m.weight.shape, generator=g) + 0.5)
                m.bias.copy_(torch.randn(m.bias.shape, generator=g) * 0.1)
            if isinstance(m, L.LayerNormMLP):
                m.layer_norm_weight.copy_(torch.rand(m.layer_norm_weight.shape, generator=g) + 0.5)
                m.layer_norm_bias.copy_(torch.randn(m.layer_norm_bias.shape, generator=g) * 0.1)
                m.fc1_weight.mul_(1.0 / (0.023 * math.sqrt(m.hidden_size)))
                m.fc2_weight.mul_(0.5 / (0.023 * math.sqrt(m.ffn_hidden_size)))
    return module


def _flash3d(case):
    """the model of a case: "plain" has one block a side and LayerNorm around pooling; "wide_scope" two blocks a side,
    scopes of 8 buckets, BatchNorm1d + GELU around pooling"""
    scope, blocks = _model_shape(case)
    chans = _channels(case)
    wide = case["shape"] == "wide_scope"
    ln = lambda c: L.LayerNorm(c)
    norm = partial(nn.BatchNorm1d, eps=1e-3, momentum=0.01) if wide else ln
    act = nn.GELU if wide else None
    spec = lambda c: [L.XFMRSpecs(c, 4 * c, c // 32, True, SwinPlan("swin", BUCKET, scope, 0), ln)] * blocks
    levels = []
    for i, c in enumerate(chans):
        last = i + 1 == len(chans)
        around = (None, None) if last else (norm, act)
        levels.append(L.F3DLevelSpecs(spec(c), spec(c), "mean", swinable_alignment(BUCKET, scope), *around, *around))
    return L.Flash3D(levels, BUCKET, scope, 2, subbuck_size=2, in_feat_dim=case["features"] or None)


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    cpu = torch.Generator().manual_seed(seed)
    torch.manual_seed(seed)
    kind = case["kind"]
    normal = lambda *shape: torch.randn(*shape, device=DEV, generator=g).to(torch.bfloat16)
    state = {"case": case}
    if kind == "attention":
        rows, h, d = case["rows"], case["heads"], case["head_dim"]
        state["qkv"] = normal(1, rows, 3 * h * d)
        state["grad"] = normal(1, rows, h, d)
        state["scopes"] = torch.arange(rows // BUCKET, dtype=torch.int32, device=DEV).view(-1, case["scope"]).view(torch.uint32)
        state["kv_len"] = None
        if case["masked"]:      # buckets three quarters to completely full
            state["kv_len"] = torch.randint(BUCKET * 3 // 4, BUCKET + 1, (rows // BUCKET,), device=DEV, generator=g,
                                            dtype=torch.int32)
        return state
    coords, seps, pts = _batch(case, g)
    state["coords"], state["seps"] = coords, seps
    if kind == "bucket":
        return state
    if kind == "stage":
        c, s = case["channels"], case["scope"]
        state["emb"] = _trained_(L.PSH3DCoordEmbedding(c, BUCKET, BUCKET * s * 6), cpu).to(DEV).eval()
        state["blk"] = _trained_(_block(c, s), cpu).to(DEV).eval()
    elif kind == "block":
        c, s = case["channels"], case["scope"]
        state["x"] = normal(_up(coords.shape[0], BUCKET * s), c)
        state["blk"] = _trained_(_block(c, s), cpu).to(DEV).eval()
    elif kind == "pool":
        # points arrive in bucket order, as pooling meets them in a model; the down features of the unpooling and the
        # gradients are those of a layer behind it
        n, c, sub = coords.shape[0], case["channels"], case["subbuck"]
        state["coords"], _ = psh_main.batch_bucket_scatter(coords, seps, BUCKET, n, 2)
        state["feat"], state["skip"] = normal(n, c).requires_grad_(), normal(n, c).requires_grad_()
        state["grad"] = normal(n, c)
        state["pool"] = L.hourglass.pooling.InbucketPoolingLayer(case["op"], BUCKET, sub)
        state["unpool"] = L.hourglass.unpool.AdditiveUnpoolLayer(sub)
    else:
        # inference runs trained weights, a training step weights near their initial values
        model = _flash3d(case).to(DEV) if case["train"] else _trained_(_flash3d(case), cpu).to(DEV)
        state["feat"] = pts if case["features"] else None
        state["model"] = model.train(case["train"])
        if case["train"]:
            if case["shape"] == "wide_scope":
                # BatchNorm on batch statistics cancels a bias in front of it: those biases are not trained
                for m in model.modules():
                    if isinstance(m, L.PoolingWrapper):
                        m.proj.bias.requires_grad_(False)
                    if isinstance(m, L.AdditiveUnpoolingWrapper):
                        m.proj[0].bias.requires_grad_(False)
                        m.proj_skip[0].bias.requires_grad_(False)
            # gradient of the loss by the model's output: a loss whose targets follow the geometry, so its gradient is a
            # smooth function of the position with some noise on it
            at = coords
            if not case["features"]:
                at, _ = psh_main.batch_bucket_scatter(coords, seps, BUCKET, _up(coords.shape[0], BUCKET * 6 * _model_shape(case)[0]), 2)
            wave = torch.randn(3, 32, device=DEV, generator=g) * 0.1
            state["grad"] = (torch.sin(at.float() @ wave) + 0.1 * normal(at.shape[0], 32)).to(torch.bfloat16)
    return state


def _block(c, scope):
    return L.XFMR(c, 4 * c, c // 32, BUCKET, True, SwinPlan("swin", BUCKET, scope, 0), lambda ch: L.LayerNorm(ch))


# ------------------------------------------------------------------------------------------------ the pass

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attention":
        b, rows, h, d = state["grad"].shape
        q, k, v = (t.view(b, rows, h, d) for t in state["qkv"].chunk(3, dim=-1))
        out, lse = torch.zeros_like(state["grad"]), torch.zeros(b, rows, h, device=DEV)
        pshattn.buck_swin_fwd(q, k, v, out, lse, state["scopes"], BUCKET, kv_len=state["kv_len"])
        dqkv, delta = torch.zeros_like(state["qkv"]), torch.zeros_like(lse)
        dq, dk, dv = (t.view(b, rows, h, d) for t in dqkv.chunk(3, dim=-1))
        pshattn.buck_swin_bwd(q, k, v, out, state["grad"], lse, delta, dq, dk, dv, state["scopes"], BUCKET,
                              kv_len=state["kv_len"])
        return {"out": out, "dqkv": dqkv}
    coords, seps = state["coords"], state["seps"]
    if kind == "bucket":
        n = coords.shape[0]
        scattered, buf = psh_main.batch_bucket_scatter(coords, seps, BUCKET, _up(n, BUCKET), case["hash"])
        return {"scattered": scattered, "id": buf.bucket_id.view(torch.int16), "count": buf.bucket_cntr.view(torch.int32),
                "slot": buf.bucket_offs.view(torch.int32)}
    if kind == "stage":
        with torch.no_grad():
            return state["blk"](None, state["emb"](coords, seps, case["hash"], lazy=True), None)
    if kind == "block":
        with torch.no_grad():
            return state["blk"](None, state["x"], None)
    if kind == "pool":
        state["feat"].grad = state["skip"].grad = None
        reduced, buf = state["pool"](coords, state["feat"], seps)
        up = state["unpool"](state["skip"], reduced, buf)
        up.backward(state["grad"])
        return {"reduced": reduced.detach(), "coord": buf.reduced_coord, "up": up.detach(), "dfeat": state["feat"].grad,
                "dskip": state["skip"].grad}
    model = state["model"]
    if not case["train"]:
        with torch.no_grad():
            out = model(coords, state["feat"], seps)
            return model.to_input_order(out) if case["features"] else out
    model.zero_grad(set_to_none=True)
    out = model(coords, state["feat"], seps)
    if case["features"]:
        out = model.to_input_order(out)
    out.backward(state["grad"])
    # the gradients as one vector, as a data-parallel program hands them to its all-reduce, and the running statistics
    grads = torch.cat([p.grad.reshape(-1) for p in model.parameters() if p.grad is not None])
    return {"out": out.detach(), "grads": grads, "stats": [b for n, b in model.named_buffers() if n.endswith(("mean", "var"))]}


# ------------------------------------------------------------------------------------------------ work and tolerance

def _block_flops(rows, c, scope, train=False, rank4=False):
    """multiply-adds count two: attention 4 T C a row (10 T C more backwards), QKV, projection and gated MLP 32 C^2 a row
    (three times that in training); rank4: QKV of a coordinate embedding, which needs only its four coefficients"""
    t = BUCKET * scope
    dense = (26 if rank4 else 32) * c * c + (24 * c if rank4 else 0)
    return rows * (4 * t * c + dense + ((10 * t * c + 2 * dense) if train else 0))


def work(case):
    kind = case["kind"]
    if kind == "attention":
        rows, h, d = case["rows"], case["heads"], case["head_dim"]
        fill = 0.875 if case["masked"] else 1.0
        return {"bytes": 2 * rows * h * d * (3 + 1 + 1 + 3), "flops": int(14 * rows * BUCKET * case["scope"] * h * d * fill ** 2)}
    n = sum(_sizes(case))
    if kind == "bucket":
        # a coordinate row in and out, bucket and slot of every point
        return {"bytes": n * (6 + 6 + 2 + 4), "flops": 0}
    if kind in ("stage", "block"):
        c, first = case["channels"], kind == "stage"
        return {"bytes": n * (2 * c + (6 if first else 2 * c)) + 2 * 16 * c * c,
                "flops": _block_flops(n, c, case["scope"], rank4=first)}
    if kind == "pool":
        c, r = case["channels"], n / case["subbuck"]
        # forward: features and skip in, sum out, pooled rows out; backward: gradient in, both gradients out
        return {"bytes": int(n * (6 + 6 * c) + r * (6 + 2 * c) + n * 6 * c), "flops": int(3 * n * c)}
    scope, blocks = _model_shape(case)
    chans, train = _channels(case), case["train"]
    flops, params, rows = 0, 0, n
    for i, c in enumerate(chans):
        flops += 2 * blocks * _block_flops(rows, c, scope, train)
        params += 2 * blocks * 16 * c * c
        if i + 1 < len(chans):
            nxt = chans[i + 1]
            # in front of pooling; skip branch and branch from below behind it
            flops += int((2 * rows * c * nxt * 2 + 2 * (rows / 2) * c * nxt) * (3 if train else 1))
            params += 3 * c * nxt
        else:
            flops += 2 * rows * c * c * (3 if train else 1)
            params += c * c
        rows = rows / 2
    moved = n * (6 + 2 * 32 + 4 * case["features"]) + 2 * params
    if train:
        moved += n * 2 * 32 + 2 * params + 4 * params      # output gradient; fp32 weights in, fp32 gradients out
    return {"bytes": int(moved), "flops": int(flops)}


def tolerance(case):
    """Measured as the distance between two correct ways through this package at the listed sizes and drawn ones: blocks
    and models with the MLP, the out-projection and the first block's embedding as separate kernels against the fused
    ones; attention and pooling against float64.  Stated: about four times what was seen."""
    kind = case["kind"]
    if kind == "bucket":
        return "exact"
    if kind == "pool":      # sums of S values in another order: a last bit of bf16 in one value of a few thousand
        return {"rel": 1e-4, "max": 0.01}
    if kind == "attention":      # 0.0029 from float64, largest 0.028
        return {"rel": 0.012, "max": 0.12}
    if kind in ("stage", "block"):      # 0.0033, largest 0.020
        return {"rel": 0.013, "max": 0.1}
    if not case["train"]:      # 0.0094 over five levels, largest 0.11
        return {"rel": 0.03, "max": 0.45}
    # outputs 0.0064, gradients 0.0035 with batch statistics; single small gradients next to large ones up to 0.65
    return {"rel": 0.026, "max": 0.9}
