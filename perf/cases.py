"""The work that users of this framework have it do, as measurable cases.

Four kinds, each through the package's Python surface (gsplat_tt_amd._lib):

frame   one view rendered by a call that is waited for (Context.render_dev into a
        GPU image, or Context.render into a host array): a preview, a thumbnail,
        an evaluation view.
path    a camera path into GPU images with frames in flight
        (Context.render_batch): video export, the orbit benchmark.
stream  a viewer's loop: each view rendered with the next one announced, images
        delivered in pinned host memory (Context.render_ring).
train   optimisation steps over a few training views (Trainer.step: forward,
        loss, backward, sparse Adam), then the updated parameters read back, as
        a program does at a checkpoint or before it edits the scene.
grads   forward and backward of one view with the gradients read back, for a
        program with an optimiser of its own.
sort    the standalone stable tile/depth sort of device keys with its per-tile
        ranges, keys and ids copied in first because the sort is in place.

Scenes follow gsplat_tt_amd/scenes.py (the box of configuration 1, the mixture
of configurations 2 and 5, the slab and shell of configuration 3, the Zipf keys
of configuration 4), drawn on the GPU because they are made often.
"""
import math

import numpy as np
import torch

from gsplat_tt_amd import _lib as L
from gsplat_tt_amd import scenes

DEV = "cuda"
TILE_BLOCK = 64  # pixels a side that the 64-bit renderings blend at once


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # a thumbnail of a small capture: launches and the wait are all of it
        _frame("frame_20k", 20_000, -1, "box", 240, 320, "f32"),
        # configuration 1, delivered to the host as a web viewer's backend does
        _frame("frame_100k_host", 100_000, -1, "box", 480, 640, "u8", host=True),
        # configuration 2: one view of a room-sized scene, full SH
        _frame("frame_1m_sh3", 1_000_000, 3, "mix", 720, 1280, "bf16"),
        # the same small scene as a path: throughput of many short frames
        _path("path_100k", 100_000, -1, "box", 480, 640, "bf16", 16),
        # configuration 3, the headline: views of an outdoor-sized scene
        _path("path_6m_sh3", 6_000_000, 3, "slab", 822, 1237, "bf16", 8),
        # an interactive viewer: odd window size, 32-pixel tiles, 8-bit images
        _stream("stream_300k_sh1", 300_000, 1, "mix", 777, 1111, "u8", 32, 6),
        # early optimisation from a sparse point cloud at a quarter resolution,
        # colours only, moments kept in bf16
        _train("train_20k", 20_000, 0, 152, 200, 10, 4, 0.0, True),
        # configuration 5: 1M Gaussians at 720p, the L1 step
        _train("train_1m_sh1", 1_000_000, 1, 720, 1280, 24, 4, 0.0, False),
        # the full 3DGS recipe: degree 3, L1 and D-SSIM, a usual image size
        _train("train_300k_sh3", 300_000, 3, 600, 800, 24, 4, 0.2, False),
        # gradients for a caller's own optimiser, odd size, full loss
        {"name": "grads_50k_sh2", "kind": "grads", "n": 50_000, "deg": 2, "scene": "mix",
         "h": 333, "w": 501, "lam": 0.2},
        # a frame's worth of keys, whole keys sorted
        {"name": "sort_2m_keys", "kind": "sort", "n": 2_000_003, "tiles": 3600, "ids": False},
        # configuration 4: 50M keys, ids and ranges wanted
        {"name": "sort_50m_ids", "kind": "sort", "n": 50_000_000, "tiles": 5000, "ids": True},
    ]


def _frame(name, n, deg, scene, h, w, out, host=False, tile=16):
    return {"name": name, "kind": "frame", "n": n, "deg": deg, "scene": scene, "h": h, "w": w,
            "out": out, "host": host, "tile": tile}


def _path(name, n, deg, scene, h, w, out, views, tile=16):
    return {"name": name, "kind": "path", "n": n, "deg": deg, "scene": scene, "h": h, "w": w,
            "out": out, "views": views, "tile": tile}


def _stream(name, n, deg, scene, h, w, out, tile, views):
    return {"name": name, "kind": "stream", "n": n, "deg": deg, "scene": scene, "h": h, "w": w,
            "out": out, "views": views, "tile": tile}


def _train(name, n, deg, h, w, steps, views, lam, bf16):
    return {"name": name, "kind": "train", "n": n, "deg": deg, "scene": "mix", "h": h, "w": w,
            "steps": steps, "views": views, "lam": lam, "bf16": bf16}


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("frame", "frame", "path", "stream", "train", "train", "grads", "sort"))
    if kind == "sort":
        return {"kind": kind, "n": size(50_000, 40_000_000), "tiles": size(300, 20_000),
                "ids": rng.random() < 0.5}
    w = size(200, 1400)
    h = max(120, int(w * rng.uniform(0.55, 0.85)))
    if kind == "train":
        c = _train("", size(20_000, 700_000), rng.randint(0, 3), h, w, rng.randint(8, 24), 4,
                   rng.choice((0.0, 0.2)), rng.random() < 0.25)
    elif kind == "grads":
        c = {"name": "", "kind": kind, "n": size(10_000, 100_000), "deg": rng.randint(0, 3),
             "scene": "mix", "h": min(h, 480), "w": min(w, 640), "lam": rng.choice((0.0, 0.2))}
    else:
        n = size(20_000, 3_000_000 if kind == "frame" else 1_500_000)
        a = (n, rng.choice((-1, 0, 1, 2, 3)), rng.choice(("box", "mix", "slab")), h, w,
             rng.choice(("u8", "bf16", "f32")))
        tile = rng.choice((16, 16, 16, 32))
        if kind == "frame":
            c = _frame("", *a, host=rng.random() < 0.3, tile=tile)
        elif kind == "path":
            c = _path("", *a, rng.randint(4, 12), tile=tile)
        else:
            c = _stream("", *a, tile, rng.randint(4, 8))
    del c["name"]
    return c


# ------------------------------------------------------------------ scenes
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _scene(case, seed):
    """Activated parameters on the GPU: means, scales, quats, opacity, colours
    (n, 3) or SH (n, K, 3)."""
    n, deg = case["n"], case["deg"]
    g = _gen(seed)
    rand = lambda *s: torch.rand(*s, generator=g, device=DEV)  # noqa: E731
    randn = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    if case["scene"] == "box":
        means = torch.stack([rand(n) * 4 - 2, rand(n) * 4 - 2, rand(n) * 6 + 2], 1)
        ls, opl = randn(n, 3) * 0.5 - 4.0, randn(n)
    elif case["scene"] == "mix":
        centers = rand(64, 3) * 10 - 5
        comp = torch.randint(64, (n,), generator=g, device=DEV)
        means = centers[comp] + randn(n, 3) * 0.5
        ls, opl = randn(n, 3) * 0.7 - 4.5, randn(n) * 1.5
    else:
        slab = int(n * 0.8)
        means = torch.empty(n, 3, device=DEV)
        means[:slab] = torch.stack([rand(slab) * 7 - 3.5, randn(slab) * 0.05,
                                    rand(slab) * 7 - 3.5], 1)
        d = randn(n - slab, 3)
        d /= d.norm(dim=1, keepdim=True)
        d[:, 1] = -d[:, 1].abs()
        means[slab:] = d * (rand(n - slab, 1) * 2 + 4.5)
        means = means[torch.randperm(n, generator=g, device=DEV)]
        ls, opl = randn(n, 3) - 5.0, randn(n) * 2.0
        big = rand(n) < 0.02
        ls = torch.where(big[:, None], randn(n, 3) * 0.5 - 2.0, ls)
    q = randn(n, 4)
    q /= q.norm(dim=1, keepdim=True)
    if deg < 0:
        col = rand(n, 3)
    else:
        col = randn(n, (deg + 1) ** 2, 3) * 0.1
        col[:, 0] = rand(n, 3)
    return {"means": means, "log_scales": ls, "quats": q, "opacity_logits": opl, "sh": col}


def _cov3d(sc):
    w, x, y, z = sc["quats"].unbind(1)
    R = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                     2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                     2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)],
                    1).view(-1, 3, 3)
    M = R * sc["log_scales"].exp()[:, None, :]
    S = (M[:, :, None, :] * M[:, None, :, :]).sum(-1)
    return S.reshape(-1, 9)


def _cameras(case, seed, count):
    """Cameras of the scene's family: (w2c, K) pairs."""
    rng = np.random.default_rng(seed)
    h, w = case["h"], case["w"]
    cams = []
    a0 = rng.uniform(0, 2 * math.pi)
    for v in range(count):
        if case["scene"] == "box":
            eye, at = rng.uniform(-0.3, 0.3, 3), np.array([0.0, 0.0, 5.0])
            f, up = w * 500.0 / 640.0, (0.0, -1.0, 0.0)
        elif case["scene"] == "mix":
            a = a0 + 2 * math.pi * v / max(count, 1)
            eye, at = np.array([6 * math.cos(a), rng.uniform(-1, 1), 6 * math.sin(a)]), np.zeros(3)
            f, up = 0.5 * w / math.tan(math.radians(25.0)), (0.0, -1.0, 0.0)
        else:
            a = a0 + 2 * math.pi * v / 64
            eye, at = np.array([4 * math.cos(a), -1.0, 4 * math.sin(a)]), np.zeros(3)
            f, up = w * 1100.0 / 1237.0, (0.0, -1.0, 0.0)
        cams.append((scenes.look_at_w2c(eye, at, up), scenes.intrinsics(f, f, 0.5 * w, 0.5 * h)))
    return cams


def _views(case, seed, count):
    return [L.make_view(e, K, case["h"], case["w"], tile_size=case.get("tile", 16),
                        output=case.get("out", "f32"))
            for e, K in _cameras(case, seed, count)]


_TORCH = {"u8": torch.uint8, "bf16": torch.bfloat16, "f32": torch.float32}


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    kind = case["kind"]
    ctx = L.Context(0)
    if kind == "sort":
        n, tiles = case["n"], case["tiles"]
        keys, ids = _sort_keys(case, seed)
        return {"kind": kind, "ctx": ctx, "case": case, "keys": keys, "ids": ids,
                "k": torch.empty_like(keys), "v": torch.empty_like(ids),
                "ranges": torch.empty(tiles, 2, dtype=torch.int32, device=DEV), "n": n}
    if kind in ("train", "grads"):
        return _prepare_train(case, seed, ctx)
    sc = _scene(case, seed)
    ctx.set_scene(sc["means"].cpu().numpy(), _cov3d(sc).cpu().numpy(),
                  torch.sigmoid(sc["opacity_logits"]).cpu().numpy(), sc["sh"].cpu().numpy(),
                  sh_degree=case["deg"])
    views = _views(case, seed, case.get("views", 1))
    state = {"kind": kind, "ctx": ctx, "views": views, "host": case.get("host", False)}
    if kind == "stream":
        ctx.out_ring_config(2 * len(views) + 1)  # the shown images and the next ones
    else:
        shape = (case["h"], case["w"], 3)
        state["outs"] = [torch.empty(shape, dtype=_TORCH[case["out"]], device=DEV) for _ in views]
        if state["host"]:
            state["outs"] = [o.cpu().numpy() for o in state["outs"]]
    return state


def _sort_keys(case, seed):
    n, tiles = case["n"], case["tiles"]
    g = _gen(seed)
    w = 1.0 / torch.arange(1, tiles + 1, device=DEV, dtype=torch.float64) ** 1.1
    cdf = torch.cumsum(w, 0)
    u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * cdf[-1]
    tile = torch.searchsorted(cdf, u).clamp_(max=tiles - 1)
    lo, hi = math.log(0.2), math.log(100.0)
    depth = torch.exp(torch.rand(n, generator=g, device=DEV) * (hi - lo) + lo)
    keys = (tile << 32) | depth.view(torch.int32).long()
    return keys, torch.arange(n, dtype=torch.int32, device=DEV)


def _train_scene(case, seed):
    """(parameters, target parameters, cameras): the target is the perturbed scene."""
    sc = _scene(case, seed)
    g = _gen(seed + 7)
    tgt = {k: v.clone() for k, v in sc.items()}
    tgt["means"] += torch.randn(tgt["means"].shape, generator=g, device=DEV) * 0.01
    tgt["sh"][:, 0] += torch.randn(tgt["means"].shape, generator=g, device=DEV) * (0.05 / 0.2820948)
    return sc, tgt, _cameras(case, seed, case.get("views", 1))


def _target_images(case, seed, views, tgt):
    ctx = L.Context(0)
    tr = L.Trainer(ctx, {k: v.cpu().numpy() for k, v in tgt.items()}, case["deg"])
    cfg = L.make_train_cfg()
    imgs = [torch.from_numpy(tr.forward(v, cfg)[0]).to(DEV) for v in views]
    ctx.close()
    return imgs


def _prepare_train(case, seed, ctx):
    sc, tgt, _ = _train_scene(case, seed)
    views = _views(case, seed, case.get("views", 1))
    targets = _target_images(case, seed, views, tgt)
    tr = L.Trainer(ctx, {k: v.cpu().numpy() for k, v in sc.items()}, case["deg"])
    if case.get("bf16"):
        tr.set_moments(True)
    if case["kind"] == "grads":
        targets = [t.cpu().numpy() for t in targets]
    return {"kind": case["kind"], "ctx": ctx, "tr": tr, "views": views, "targets": targets,
            "steps": case.get("steps", 1), "cfg": L.make_train_cfg(lambda_dssim=case["lam"])}


# ------------------------------------------------------------------ run
def run(s):
    kind, ctx = s["kind"], s["ctx"]
    if kind == "frame":
        if s["host"]:
            return ctx.render(s["views"][0], out=s["outs"][0])[0]
        ctx.render_dev(s["views"][0], s["outs"][0].data_ptr())
        return s["outs"][0]
    if kind == "path":
        ctx.render_batch(s["views"], [o.data_ptr() for o in s["outs"]])
        return s["outs"]
    if kind == "stream":
        v = s["views"]
        return [ctx.render_ring(v[i], v[i + 1] if i + 1 < len(v) else None)[0]
                for i in range(len(v))]
    if kind == "train":
        losses = []
        for k in range(s["steps"]):
            i = k % len(s["views"])
            losses.append(s["tr"].step(s["views"][i], s["cfg"], s["targets"][i].data_ptr(),
                                       target_on_device=True)["loss"])
        return {"losses": np.array(losses), "params": s["tr"].read(0)}
    if kind == "grads":
        img, T, _, st = s["tr"].forward(s["views"][0], s["cfg"], s["targets"][0])
        s["tr"].backward(s["cfg"])
        return {"image": img, "T": T, "loss": st["loss"], "grads": s["tr"].read(3)}
    n = s["n"]
    ctx.d2d(s["k"].data_ptr(), s["keys"].data_ptr(), 8 * n)
    ctx.d2d(s["v"].data_ptr(), s["ids"].data_ptr(), 4 * n)
    tiles = s["ranges"].shape[0]
    if s["case"]["ids"]:
        ctx.sort_tile_depth_ids_dev(s["k"].data_ptr(), s["v"].data_ptr(), n, tiles,
                                    s["ranges"].data_ptr(), num_gaussians=n)
        return s["v"], s["ranges"]
    ctx.sort_tile_depth_dev(s["k"].data_ptr(), s["v"].data_ptr(), n, tiles,
                            s["ranges"].data_ptr())
    return s["k"], s["v"], s["ranges"]


# ------------------------------------------------------------------ work
def work(case):
    """Inputs read once and outputs written once per frame or step. About half of
    a scene's Gaussians are visible in a view; a pixel blends on the order of
    100 of them (20 operations each, three times that with the backward)."""
    kind, n = case["kind"], case["n"]
    if kind == "sort":
        moved = 12 + (4 if case["ids"] else 12)
        return {"bytes": n * (moved + 24) + 8 * case["tiles"], "flops": 0}
    px = case["h"] * case["w"]
    K = (max(case["deg"], 0) + 1) ** 2
    if kind in ("train", "grads"):
        planes = 11 + 3 * K
        steps = case.get("steps", 1)
        mom = 2 if case.get("bf16") else 4
        step = n * planes * 4 + px * 24
        if kind == "train":  # visible rows: both moments and the parameters, in and out
            step += n // 2 * planes * (8 + 4 * mom)
        else:
            step += n * planes * 4
        return {"bytes": steps * step + n * planes * 4,
                "flops": steps * (px * 100 * 60.0 + n * 600.0)}
    views = case.get("views", 1)
    e = {"u8": 1, "bf16": 2, "f32": 4}[case["out"]]
    per = n * 40 + n // 2 * 12 * K + px * 3 * e
    return {"bytes": views * per, "flops": views * (px * 100 * 20.0 + n * 200.0)}


def tolerance(case):
    kind = case["kind"]
    if kind == "sort":
        return "exact"
    if kind == "grads":
        # a rounding of alpha takes a pixel over the 1/255 threshold or not: against
        # 64 bits the gradients are up to 1e-3 off for that
        return {"rel": 4e-3, "max": 0.3}
    if kind == "train":
        # Adam turns a gradient that cancels to nothing into a whole step of
        # either sign, so single values may be a few steps apart (two runs of the
        # same 24 steps differ by up to 1.8e-3)
        return {"rel": 8e-3, "max": 0.9}
    if case["out"] == "f32":
        return {"rel": 3e-5, "max": 0.02}
    if case["out"] == "bf16":
        return {"rel": 4e-3, "max": 0.04}
    return {"rel": 0.0, "max": 0.0, "differ": 0.005}


# ------------------------------------------------------------------ 64 bits
def exact(case, seed):
    kind = case["kind"]
    if kind == "sort" or case.get("out") == "u8":
        return None  # whole numbers
    blocks = math.ceil(case["h"] / TILE_BLOCK) * math.ceil(case["w"] / TILE_BLOCK)
    if kind == "grads" or kind == "train":
        if blocks * case.get("steps", 1) > 4000 or case["n"] > 400_000:
            return None
        return _exact_train(case, seed)
    if case["n"] * case.get("views", 1) > 4_000_000:
        return None
    sc = {k: v.double() for k, v in _scene(case, seed).items()}
    cov = _cov3d(_scene(case, seed)).double().view(-1, 3, 3)
    out = [_exact_frame(case, sc, cov, e, K)
           for e, K in _cameras(case, seed, case.get("views", 1))]
    return out[0] if kind == "frame" else out


def _camera64(e, K):
    e = torch.tensor(np.asarray(e, np.float32), device=DEV, dtype=torch.float64)
    return e[:3, :3], e[:3, 3], float(K[0, 0]), float(K[1, 1]), float(K[0, 2]), float(K[1, 2])


def _basis(d, deg):
    x, y, z = d.unbind(1)
    xx, yy, zz = x * x, y * y, z * z
    b = [torch.full_like(x, 0.28209479177387814)]
    if deg >= 1:
        b += [-0.4886025119029199 * y, 0.4886025119029199 * z, -0.4886025119029199 * x]
    if deg >= 2:
        b += [1.0925484305920792 * x * y, -1.0925484305920792 * y * z,
              0.31539156525252005 * (2 * zz - xx - yy), -1.0925484305920792 * x * z,
              0.5462742152960396 * (xx - yy)]
    if deg >= 3:
        b += [-0.5900435899266435 * y * (3 * xx - yy), 2.890611442640554 * x * y * z,
              -0.4570457994644658 * y * (4 * zz - xx - yy),
              0.3731763325901154 * z * (2 * zz - 3 * xx - 3 * yy),
              -0.4570457994644658 * x * (4 * zz - xx - yy), 1.445305721320277 * z * (xx - yy),
              -0.5900435899266435 * x * (xx - 3 * yy)]
    return torch.stack(b, 1)


def _project64(means, cov, e, K, near, lowpass):
    """Camera-space z, 2D centres and low-passed 2D covariances (a, b, c)."""
    R, t, fx, fy, cx, cy = _camera64(e, K)
    x, y, z = (means @ R.T + t).unbind(1)
    ok = z > near
    zs = torch.where(ok, z, torch.ones_like(z))
    zero = torch.zeros_like(zs)
    J = torch.stack([fx / zs, zero, -fx * x / zs ** 2, zero, fy / zs, -fy * y / zs ** 2],
                    1).view(-1, 2, 3)
    Tm = J @ R
    c2 = (Tm @ cov) @ Tm.transpose(1, 2)
    return (z, ok, fx * x / zs + cx, fy * y / zs + cy, c2[:, 0, 0] + lowpass, c2[:, 0, 1],
            c2[:, 1, 1] + lowpass)


def _colours64(means, sh, e, K, deg):
    R, t, *_ = _camera64(e, K)
    d = means - (-R.T @ t)
    d = d / d.norm(dim=1, keepdim=True)
    return (_basis(d, deg)[:, :, None] * sh).sum(1) + 0.5


def _exact_frame(case, sc, cov, e, K):
    """The view by the render rules: rectangles of whole tiles, alpha at most 0.99,
    a microblock of 8 x 4 pixels stopping once all of it is below 1/255. (The
    culls' floor of 2^-14 and the stop's four-entry steps are left out.)"""
    h, w, ts = case["h"], case["w"], case["tile"]
    thr = 1.0 / 255.0
    z, ok, u, v, a, b, c = _project64(sc["means"], cov, e, K, 0.2, 0.3)
    op = torch.sigmoid(sc["opacity_logits"])
    k = torch.sqrt(2 * torch.log((op * 16384.0).clamp(min=1.0))).clamp(max=3.0)
    rx, ry = torch.ceil(k * a.clamp(min=0).sqrt()), torch.ceil(k * c.clamp(min=0).sqrt())
    rmax = min(h, w) // 2
    ok &= (op >= thr) & (rx > 0) & (ry > 0) & (rx <= rmax) & (ry <= rmax)
    ok &= (u + rx > 0) & (u - rx < w) & (v + ry > 0) & (v - ry < h)
    idx = torch.nonzero(ok)[:, 0]
    idx = idx[torch.argsort(z[idx], stable=True)]
    u, v, a, b, c, op, rx, ry = (q[idx] for q in (u, v, a, b, c, op, rx, ry))
    det = (a * c - b * b).clamp(min=1e-6)
    A, B, C = c / det, -b / det, a / det
    col = sc["sh"][idx]
    if case["deg"] >= 0:
        col = _colours64(sc["means"][idx], col, e, K, case["deg"])
        col = col.clamp(0.0, 1.0)
    tx, ty = math.ceil(w / ts) - 1, math.ceil(h / ts) - 1
    x0, x1 = ((u + s * rx).div(ts).trunc().clamp(0, tx) for s in (-1, 1))
    y0, y1 = ((v + s * ry).div(ts).trunc().clamp(0, ty) for s in (-1, 1))
    img = torch.zeros(h, w, 3, device=DEV, dtype=torch.float64)
    B_ = TILE_BLOCK
    for by in range(0, h, B_):
        for bx in range(0, w, B_):
            sel = torch.nonzero((x1 * ts + ts > bx) & (x0 * ts < bx + B_) &
                                (y1 * ts + ts > by) & (y0 * ts < by + B_))[:, 0]
            py, px = torch.meshgrid(torch.arange(by, by + B_, device=DEV),
                                    torch.arange(bx, bx + B_, device=DEV), indexing="ij")
            T = torch.ones(B_, B_, device=DEV, dtype=torch.float64)
            acc = torch.zeros(3, B_, B_, device=DEV, dtype=torch.float64)
            inside = (px < w) & (py < h)
            tpx, tpy = (px // ts).double(), (py // ts).double()
            for s in sel.split(2048):
                q = lambda t: t[s][:, None, None]  # noqa: E731
                dx, dy = px + 0.5 - q(u), py + 0.5 - q(v)
                power = -0.5 * (q(A) * dx * dx + 2 * q(B) * dx * dy + q(C) * dy * dy)
                al = (q(op) * torch.exp(power.clamp(max=0.0))).clamp(max=0.99)
                al = al * ((tpx >= q(x0)) & (tpx <= q(x1)) & (tpy >= q(y0)) & (tpy <= q(y1)))
                cum = torch.cumprod(1 - al, 0) * T
                before = torch.cat([T[None], cum[:-1]])
                blocks = (before * inside).view(-1, B_ // 4, 4, B_ // 8, 8).amax((2, 4))
                alive = (blocks >= thr).repeat_interleave(4, 1).repeat_interleave(8, 2)
                acc += torch.einsum("nc,nyx->cyx", col[s], al * before * alive)
                T = cum[-1]
                if not bool(alive[-1].any()):
                    break
            hh, ww = min(B_, h - by), min(B_, w - bx)
            img[by:by + hh, bx:bx + ww] = acc[:, :hh, :ww].permute(1, 2, 0)
    return img


def _blend_block(px, py, p):
    """Training rules over one block: colours (3, y, x) and transmittance."""
    u, v, A, B, C, op, col = p
    q = lambda t: t[:, None, None]  # noqa: E731
    dx, dy = px - q(u), py - q(v)
    power = -0.5 * (q(A) * dx * dx + 2 * q(B) * dx * dy + q(C) * dy * dy)
    al = (q(op) * torch.exp(power.clamp(max=0.0))).clamp(max=0.99)
    al = torch.where(al >= 1.0 / 255.0, al, torch.zeros_like(al))
    with torch.no_grad():
        live = torch.cumprod(1 - al, 0) >= 1e-4
    al = al * live
    cum = torch.cumprod(1 - al, 0)
    before = torch.cat([torch.ones_like(cum[:1]), cum[:-1]])
    return torch.einsum("nc,nyx->cyx", col, al * before), cum[-1]


def _train_loss(img, tgt, lam):
    l1 = (img - tgt).abs().mean()
    if lam == 0.0:
        return l1
    g = torch.exp(-((torch.arange(11, device=DEV, dtype=torch.float64) - 5) ** 2) / 4.5)
    g = g / g.sum()
    win = (g[:, None] * g[None, :]).expand(3, 1, 11, 11).contiguous()
    x, y = img.permute(2, 0, 1)[None], tgt.permute(2, 0, 1)[None]

    def f(t):
        t = torch.nn.functional.pad(t, (5, 5, 5, 5)).unfold(2, 11, 1).unfold(3, 11, 1)
        return (t * win[:, 0][None, :, None, None]).sum((-1, -2))

    mx, my = f(x), f(y)
    cxx, cyy, cxy = f(x * x) - mx * mx, f(y * y) - my * my, f(x * y) - mx * my
    S = ((2 * mx * my + 1e-4) * (2 * cxy + 9e-4)) / \
        ((mx * mx + my * my + 1e-4) * (cxx + cyy + 9e-4))
    return (1 - lam) * l1 + lam * (1 - S.mean())


def _forward_backward(par, tgt, cam, case):
    """(image, T, loss, gradients, rows the sparse optimiser updates)."""
    h, w, deg = case["h"], case["w"], case["deg"]
    e, K = cam
    p = {k: t.detach().requires_grad_(True) for k, t in par.items()}
    qn = p["quats"] / p["quats"].norm(dim=1, keepdim=True)
    cov = _cov3d({"quats": qn, "log_scales": p["log_scales"]}).view(-1, 3, 3)
    z, ok, u, v, a, b, c = _project64(p["means"], cov, e, K, 0.2, 0.3)
    op = torch.sigmoid(p["opacity_logits"])
    col = _colours64(p["means"], p["sh"], e, K, deg).clamp(min=0.0)
    det = a * c - b * b
    flat = [u, v, c / det, -b / det, a / det, op, col]
    with torch.no_grad():
        r3x, r3y = torch.ceil(3 * a.clamp(min=0).sqrt()), torch.ceil(3 * c.clamp(min=0).sqrt())
        vis = ok & (u + r3x > 0) & (u - r3x < w) & (v + r3y > 0) & (v - r3y < h)
        use = ok & (op >= 1.0 / 255.0) & (det > 0)
        k = torch.sqrt(2 * torch.log((op * 255.0).clamp(min=1.0)))
        rx, ry = k * a.clamp(min=0).sqrt() + 1, k * c.clamp(min=0).sqrt() + 1
        use &= (u + rx > 0) & (u - rx < w) & (v + ry > 0) & (v - ry < h)
        idx = torch.nonzero(use)[:, 0]
        idx = idx[torch.argsort(z[idx], stable=True)]
        rx, ry, ui, vi = rx[idx], ry[idx], u[idx], v[idx]
        leaf = [t.detach()[idx] for t in flat]
        grad = [torch.zeros_like(t) for t in leaf]
        img = torch.zeros(h, w, 3, device=DEV, dtype=torch.float64)
        Tf = torch.ones(h, w, device=DEV, dtype=torch.float64)
        blocks = []
        for by in range(0, h, TILE_BLOCK):
            for bx in range(0, w, TILE_BLOCK):
                hh, ww = min(TILE_BLOCK, h - by), min(TILE_BLOCK, w - bx)
                s = torch.nonzero((ui + rx > bx) & (ui - rx < bx + ww) & (vi + ry > by) &
                                  (vi - ry < by + hh))[:, 0]
                if s.numel() == 0:
                    continue
                py, px = torch.meshgrid(torch.arange(by, by + hh, device=DEV) + 0.5,
                                        torch.arange(bx, bx + ww, device=DEV) + 0.5,
                                        indexing="ij")
                blocks.append((by, bx, hh, ww, s, px.double(), py.double()))
                o, T = _blend_block(px.double(), py.double(), [t[s] for t in leaf])
                img[by:by + hh, bx:bx + ww] = o.permute(1, 2, 0)
                Tf[by:by + hh, bx:bx + ww] = T
    im = img.clone().requires_grad_(True)
    loss = _train_loss(im, tgt, case["lam"])
    dimg, = torch.autograd.grad(loss, im)
    for by, bx, hh, ww, s, px, py in blocks:
        q = [t[s].requires_grad_(True) for t in leaf]
        o, _ = _blend_block(px, py, q)
        gs = torch.autograd.grad(o, q, dimg[by:by + hh, bx:bx + ww].permute(2, 0, 1))
        for acc, t in zip(grad, gs):
            acc.index_add_(0, s, t)
    names = list(p)
    g = torch.autograd.grad([t[idx] for t in flat], [p[k] for k in names], grad,
                            allow_unused=True)
    grads = {k: (torch.zeros_like(p[k]) if t is None else t)
             for k, t in zip(names, g)}
    return img, Tf, float(loss), grads, vis


def _exact_train(case, seed):
    sc, tgt, cams = _train_scene(case, seed)
    par = {k: v.double() for k, v in sc.items()}
    targets = [t.double() for t in _target_images(case, seed, _views(case, seed, len(cams)), tgt)]
    if case["kind"] == "grads":
        img, T, loss, grads, _ = _forward_backward(par, targets[0], cams[0], case)
        return {"image": img, "T": T, "loss": loss, "grads": grads}
    lr = {"means": 1.6e-4, "log_scales": 5e-3, "quats": 1e-3, "opacity_logits": 0.05}
    m = {k: torch.zeros_like(v) for k, v in par.items()}
    v2 = {k: torch.zeros_like(v) for k, v in par.items()}
    keep = (lambda t: t.to(torch.bfloat16).double()) if case["bf16"] else (lambda t: t)
    losses = []
    for k in range(case["steps"]):
        i = k % len(cams)
        _, _, loss, grads, vis = _forward_backward(par, targets[i], cams[i], case)
        losses.append(loss)
        for name, g in grads.items():
            rate = lr.get(name)
            if rate is None:  # SH: the constant term's rate, then a twentieth
                rate = torch.full((1, g.shape[1], 1), 2.5e-3 / 20, device=DEV,
                                  dtype=torch.float64)
                rate[:, 0] = 2.5e-3
            mn = 0.9 * m[name] + 0.1 * g
            vn = 0.999 * v2[name] + 0.001 * g * g
            step = rate / (1 - 0.9 ** (k + 1)) * mn / \
                (vn.sqrt() / math.sqrt(1 - 0.999 ** (k + 1)) + 1e-15)
            row = vis.view(-1, *([1] * (g.dim() - 1)))
            par[name] = torch.where(row, par[name] - step, par[name])
            m[name] = torch.where(row, keep(mn), m[name])
            v2[name] = torch.where(row, keep(vn), v2[name])
    return {"losses": np.array(losses), "params": par}
