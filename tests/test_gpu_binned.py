"""The ways a frame's tile lists are made: binned (pairs counted per tile, each
list sorted on its own in runs of 2048), by blocks (depth sort, items of 4 x 4 tiles
sorted by block and split) and sorted (depth sort, then tile sort; the microblock
statistics select it). All give the stable (tile, depth bits, compact id)
order, so ids, ranges, counts and images are compared for equality, at list lengths
around the runs of the list sort, with equal depths, empty views and many tiles."""
import ctypes

import numpy as np
import pytest

from gsplat_tt_amd import _lib as L
from gsplat_tt_amd import scenes

pytestmark = pytest.mark.gpu


def _both(ctx, view):
    """(image, stats, readback) of the view, binned then sorted."""
    out = []
    for stats in (False, True):
        ctx.set_cull_stats(stats)
        img, st = ctx.render(view)
        out.append((img, st, ctx.frame_readback() if st["num_visible"] else None))
    ctx.set_cull_stats(False)
    return out


def _equal(a, b):
    assert np.array_equal(a[0], b[0])
    for k in ("num_visible", "num_entries", "pairs_pre"):
        assert a[1][k] == b[1][k], k
    if a[2] is not None:
        assert np.array_equal(a[2]["tile_ranges"], b[2]["tile_ranges"])
        assert np.array_equal(a[2]["sorted_ids"], b[2]["sorted_ids"])


def _stack(n, levels, spread=0.004, seed=0):
    """n small Gaussians in one column at z of a few levels (many equal depths)."""
    rng = np.random.default_rng(seed)
    z = (2.0 + rng.integers(0, levels, n) / 64.0).astype(np.float32)
    means = np.stack([rng.normal(0, spread, n) * z, rng.normal(0, spread, n) * z, z], 1)
    q = rng.standard_normal((n, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    cov = scenes.cov3d(np.full((n, 3), 0.004, np.float32), q.astype(np.float32))
    return (means.astype(np.float32), cov, rng.uniform(0.05, 0.6, n).astype(np.float32),
            rng.random((n, 3)).astype(np.float32))


@pytest.mark.parametrize("n,levels", [(1, 1), (7, 2), (8, 1), (9, 3), (64, 2), (513, 5),
                                      (2047, 40), (2048, 1), (2049, 7), (4097, 500), (9000, 3)])
def test_lists_around_the_runs(gpu_ctx, n, levels):
    print("lists", n, levels, flush=True)
    gpu_ctx.set_scene(*_stack(n, levels, seed=n))
    for ts, h, w in ((16, 48, 64), (32, 35, 61)):
        K = scenes.intrinsics(60, 60, w / 2, h / 2)
        view = L.make_view(np.eye(4, dtype=np.float32), K, h, w, tile_size=ts, output="f32")
        a, b = _both(gpu_ctx, view)
        if n == 9000:
            r = a[2]["tile_ranges"]
            assert (r[:, 1] - r[:, 0]).max() > 4096  # a list of several runs
        _equal(a, b)


@pytest.mark.parametrize("n,deg", [(511, 0), (512, 1), (1025, 2), (1 << 18, 3), (1 << 18, -1),
                                   ((1 << 18) + 1, 2)])
def test_projection_partitions(gpu_ctx, n, deg):
    """Binned projection by one and by four Gaussians a thread (the line is at 2^18)
    against the sorted frames', at whole and ragged partitions and every colour form."""
    print("partitions", n, deg, flush=True)
    rng = np.random.default_rng(n)
    means, cov, op, col = _stack(n, 300, spread=0.3, seed=n)
    means[:, 2] *= np.where(rng.random(n) < 0.2, -1, 1)  # a fifth behind the camera
    if deg >= 0:
        col = rng.uniform(-0.5, 0.5, (n, (deg + 1) ** 2, 3)).astype(np.float32)
    gpu_ctx.set_scene(means, cov, op, col, sh_degree=deg)
    K = scenes.intrinsics(200, 200, 120, 67)
    view = L.make_view(np.eye(4, dtype=np.float32), K, 135, 241, tile_size=16, output="f32")
    a, b = _both(gpu_ctx, view)
    assert a[1]["num_visible"] > n // 2
    _equal(a, b)


@pytest.mark.parametrize("h,w,ts,n,spread", [
    (129 * 16, 128 * 16 + 1, 16, 9000, 0.004),   # a block's list of five segments
    (203 * 16 - 7, 131 * 16, 16, 3000, 0.3), (16, 16390 * 16 - 9, 16, 700, 0.3),
    (16390 * 16 - 9, 5, 16, 2049, 0.3), (129 * 32 - 31, 130 * 32, 32, 2000, 0.2),
    (200, 299, 16, (1 << 20) + 1, 0.1), (33, 17, 32, (1 << 20) + 7, 0.002)])  # one sort pass
@pytest.mark.parametrize("cull", [True, False])
def test_lists_by_blocks(gpu_ctx, h, w, ts, n, spread, cull):
    """Frames of more than 2^14 tiles, and first frames of more than 2^20 Gaussians,
    are made by blocks: whole and cut blocks, one row or column of them, one block
    and thousands, lists of several segments, with and without the tile cull."""
    print("blocks", h, w, ts, n, cull, flush=True)
    if not cull and n > 9000:
        n = (1 << 20) + 3
    gpu_ctx.set_scene(*_stack(n, 300, spread=spread, seed=n))
    K = scenes.intrinsics(0.5 * w, 0.5 * h, w / 2, h / 2)
    view = L.make_view(np.eye(4, dtype=np.float32), K, h, w, tile_size=ts, output="u8",
                       cull_disabled=not cull, max_radius=-1)
    a, b = _both(gpu_ctx, view)
    assert a[1]["num_visible"] > n // 3
    _equal(a, b)


def test_blocks_pair_limit():
    """The pair limit counts candidate tiles, not items: the same floor, retries and
    image by blocks as sorted."""
    print("block limit", flush=True)
    scene, cams = scenes.config1(seed=5, n=6_000)
    cov = scenes.cov3d(scene.scales, scene.quats)
    h, w = 130 * 16 - 15, 129 * 16
    K = scenes.intrinsics(500 * w / 640, 500 * w / 640, w / 2, h / 2)
    ctx = L.Context(0)
    try:
        ctx.set_scene(scene.means, cov, scene.opacities, scene.colors)
        view = L.make_view(cams[0].w2c, K, h, w, tile_size=16, output="bf16")
        full = ctx.render(view)[1]["pairs_pre"]
        ctx.set_pair_limit(int(full * 0.9))
        a, b = _both(ctx, view)
        assert a[1]["floor_retries"] == b[1]["floor_retries"] > 0
        assert a[1]["contrib_floor"] == b[1]["contrib_floor"]
        _equal(a, b)
    finally:
        ctx.close()


def test_training_forward_by_blocks(gpu_ctx):
    """A training image of more than 2^14 tiles (by blocks) against the same view two
    rows of tiles shorter (binned): the shared rows are the same bit for bit."""
    print("train blocks", flush=True)
    n, w = 4000, 129 * 16 - 3
    rng = np.random.default_rng(3)
    z = rng.uniform(2, 4, n)
    p = {"means": np.stack([rng.uniform(-0.5, 0.5, n) * z, rng.uniform(-0.5, 0.5, n) * z, z], 1),
         "log_scales": rng.normal(-3.5, 0.5, (n, 3)), "quats": rng.standard_normal((n, 4)),
         "opacity_logits": rng.normal(0, 1.0, n), "sh": rng.uniform(-0.5, 0.5, (n, 4, 3))}
    p = {k: v.astype(np.float32) for k, v in p.items()}
    K = scenes.intrinsics(0.9 * w, 0.9 * w, w / 2, 64 * 16)
    tr = L.Trainer(gpu_ctx, p, 1)
    imgs = []
    for rows in (127, 129):
        view = L.make_view(np.eye(4, dtype=np.float32), K, rows * 16, w, tile_size=16)
        imgs.append(tr.forward(view, L.make_train_cfg())[0])
    assert imgs[0].any() and np.array_equal(imgs[1][:127 * 16], imgs[0])


def test_many_tiles_and_empty_views(gpu_ctx):
    """Close to the most tiles of a binned frame (127 x 129 = 16383 of 16384), one row of
    tiles past it (sorted either way), and a view with nothing visible."""
    print("many tiles", flush=True)
    scene, cams = scenes.config1(seed=5, n=6_000)
    cov = scenes.cov3d(scene.scales, scene.quats)
    gpu_ctx.set_scene(scene.means, cov, scene.opacities, scene.colors)
    for h, w in ((127 * 16, 129 * 16 - 3), (130 * 16 - 15, 129 * 16)):
        K = scenes.intrinsics(500 * w / 640, 500 * w / 640, w / 2, h / 2)
        view = L.make_view(cams[0].w2c, K, h, w, tile_size=16, output="bf16")
        _equal(*_both(gpu_ctx, view))
    back = np.diag([-1, 1, -1, 1]).astype(np.float32)
    view = L.make_view(back, cams[0].K, 100, 120, tile_size=16, output="f32")
    a, b = _both(gpu_ctx, view)
    assert a[1]["num_visible"] == b[1]["num_visible"] == 0 and not a[0].any() and not b[0].any()


def test_plan_follows_the_pairs():
    """A scene whose view has more pairs than binning pays for goes on sorted, one with
    fewer binned again: every frame of the change equals the sorted one."""
    print("plan", flush=True)
    scene, cams = scenes.config3(seed=17, n=700_000, views=3)
    cov = scenes.cov3d(scene.scales, scene.quats)
    ctx = L.Context(0)
    try:
        ctx.set_scene(scene.means, cov, scene.opacities, scene.sh, sh_degree=3)
        near = [L.make_view(c.w2c, c.K, c.height, c.width, tile_size=16, output="bf16")
                for c in cams]
        far_w2c = cams[0].w2c.copy()
        far_w2c[2, 3] += 60.0  # small on screen: few pairs
        far = L.make_view(far_w2c, cams[0].K, cams[0].height, cams[0].width, tile_size=16,
                          output="bf16")
        pairs = []
        for view in (near[0], near[1], far, far, near[2], far):
            a, st = ctx.render(view)
            rb = ctx.frame_readback()
            pairs.append(st["num_entries"])
            _equal((a, st, rb), _both(ctx, view)[1])
        assert max(pairs) > 2_400_000 and min(pairs) < 1_800_000, pairs
        outs = [np.empty((822, 1237, 3), np.uint16) for _ in range(6)]
        views = [near[0], far, near[1], far, near[2], far]
        ctx.render_batch(views, outs, out_on_device=False)
        for v, o in zip(views, outs):
            assert np.array_equal(o, _both(ctx, v)[1][0])
    finally:
        ctx.close()


@pytest.mark.parametrize("h,w,ts", [(1, 1, 16), (4, 8, 16), (5, 9, 32), (3, 7, 16), (17, 33, 16),
                                    (35, 61, 32), (64, 48, 16)])
@pytest.mark.parametrize("n,op", [(3, 0.9), (70, 0.03), (67, 0.5), (400, 0.15), (400, 0.98)])
def test_blend_by_microblock_equals_by_band(gpu_ctx, h, w, ts, n, op):
    """render() blends with a wave per microblock, gs_cull_and_blend with one per band:
    the same image bit for bit, for whole and cut microblocks, lists whose kept entries
    leave every remainder of four, faint entries (no early-out) and opaque ones."""
    print("blend", h, w, ts, n, op, flush=True)
    rng = np.random.default_rng(n + h)
    f = 0.7 * max(h, w)
    z = rng.uniform(2, 4, n)
    means = np.stack([rng.uniform(-0.6, 0.6, n) * w / f * z, rng.uniform(-0.6, 0.6, n) * h / f * z,
                      z], 1).astype(np.float32)
    q = rng.standard_normal((n, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    cov = scenes.cov3d(np.exp(rng.normal(-1.5, 0.8, (n, 3))).astype(np.float32),
                       q.astype(np.float32))
    opac = np.full(n, op, np.float32)
    col = rng.random((n, 3)).astype(np.float32)
    view = L.make_view(np.eye(4, dtype=np.float32), scenes.intrinsics(f, f, w / 2, h / 2), h, w,
                       tile_size=ts, output="f32", max_radius=10_000)
    gpu_ctx.set_scene(means, cov, opac, col)
    img, st = gpu_ctx.render(view)
    p = gpu_ctx.project(means, cov, opac, col, view)
    g, t, _ = gpu_ctx.tile_assign(p["means2d"], p["radii"], h, w, ts, p["covs2d"],
                                  p["opacities"])
    assert g.shape[0] == st["num_entries"]
    if g.shape[0] == 0:
        assert not img.any()
        return
    ids, ranges = gpu_ctx.sort_and_bin(g, t, p["depths"], -(-w // ts), -(-h // ts))
    ref = gpu_ctx.cull_and_blend(p["means2d"], p["covs2d"], p["colors"], p["opacities"], ids,
                                 ranges, view)
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("h,w,ts", [(48, 64, 16), (32 * 16, 64 * 16, 16), (33 * 16, 64 * 16, 16),
                                    (64 * 16, 64 * 16 - 3, 16), (65 * 16 - 5, 64 * 16, 16),
                                    (480, 640, 32), (32 * 32, 32 * 32, 32), (33 * 32, 32 * 32, 32),
                                    (96 * 16, 64 * 16, 16), (97 * 16, 64 * 16, 16)])
def test_blend_of_frames_in_flight(h, w, ts):
    """A wave per microblock blends up to 8192 bands of 16 x 4 pixels (frames in flight,
    16384 binned ones) or 24576 (alone), a wave per band above: the images of a path are
    those of single frames on both sides of each line, binned and not (more than 2^20
    Gaussians), through captures and replays."""
    print("blend in flight", h, w, ts, flush=True)
    for n in (3000, (1 << 20) + 5):
        ctx = L.Context(0)
        try:
            ctx.set_scene(*_stack(n, 300, spread=0.25, seed=n + h))
            views = []
            for k in range(6):
                w2c = np.eye(4, dtype=np.float32)
                w2c[0, 3] = 0.03 * k
                views.append(L.make_view(w2c, scenes.intrinsics(0.7 * w, 0.7 * w, w / 2, h / 2),
                                         h, w, tile_size=ts, output="bf16"))
            ref = [ctx.render(v)[0].copy() for v in views]
            for _ in range(2):
                outs = [np.empty((h, w, 3), np.uint16) for _ in views]
                ctx.render_batch(views, outs, out_on_device=False)
                assert all(np.array_equal(a, b) for a, b in zip(ref, outs))
        finally:
            ctx.close()


@pytest.mark.parametrize("n", [12_000, 30_000, 120_000])
@pytest.mark.parametrize("h,w,ts", [(16, 16, 16), (33, 17, 16), (40, 60, 32)])
def test_long_lists(n, h, w, ts):
    """Lists of many runs, in one tile or a few: the frames on the way from the first
    guess to the way that the longest list asks for equal the sorted ones, also after a
    view of the same size with short lists."""
    print("long lists", n, h, w, ts, flush=True)
    ctx = L.Context(0)
    try:
        ctx.set_scene(*_stack(n, 500, spread=0.02, seed=n))
        K = scenes.intrinsics(60, 60, w / 2, h / 2)
        near = L.make_view(np.eye(4, dtype=np.float32), K, h, w, tile_size=ts, output="f32")
        aside = np.eye(4, dtype=np.float32)
        aside[0, 3] = -50.0  # nothing in view
        away = L.make_view(aside, K, h, w, tile_size=ts, output="f32")
        for view in (near, near, away, away, near, near):
            a, st = ctx.render(view)
            rb = ctx.frame_readback() if st["num_visible"] else None
            _equal((a, st, rb), _both(ctx, view)[1])
        assert (rb["tile_ranges"][:, 1] - rb["tile_ranges"][:, 0]).max() > 2 * 2048
    finally:
        ctx.close()


def _free_bytes(ctx):
    """Free device memory, by the HIP runtime that the library is linked to."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctx._L.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_more_candidates_than_a_binned_frame_holds():
    """A view of 29M candidates over 14400 tiles and an empty one by turns, alone, in paths and
    in training: a binned frame that has no room for its candidates is made again and
    equals the sorted one, and its bins are allocated for 2^22 candidates (about 64 MB), not
    for the pair capacity (460 MB): the context takes four buffers of that capacity
    (32.4M, 4 bytes), 64 MB of bins and some 70 MB of others, below 800 MB."""
    print("binned room", flush=True)
    rng = np.random.default_rng(8)
    n, h, w, f = 2000, 1440, 2560, 2000.0
    means = np.concatenate([rng.normal(0, 0.01, (n, 2)), rng.uniform(2, 3, (n, 1))], 1)
    q = np.tile(np.float32([1, 0, 0, 0]), (n, 1))
    scale = np.full((n, 3), 2.0, np.float32)
    views = []
    for turn in (1, -1):  # the second looks away
        w2c = np.diag([turn, 1, turn, 1]).astype(np.float32)
        views.append(L.make_view(w2c, scenes.intrinsics(f, f, w / 2, h / 2), h, w, tile_size=16,
                                 output="bf16", max_radius=100_000))
    near, away = views
    ctx = L.Context(0)
    try:
        ctx.set_scene(means.astype(np.float32), scenes.cov3d(scale, q),
                      rng.uniform(0.01, 0.05, n).astype(np.float32),
                      rng.random((n, 3)).astype(np.float32))
        free = _free_bytes(ctx)
        a, b = _both(ctx, near)
        assert a[1]["pairs_pre"] == n * 14400
        _equal(a, b)
        away_img = ctx.render(away)[0].copy()
        for _ in range(3):
            assert np.array_equal(ctx.render(away)[0], away_img)
            img, st = ctx.render(near)
            assert np.array_equal(img, a[0]) and st["pairs_pre"] == a[1]["pairs_pre"]
            ctx.render(away)
        used = free - _free_bytes(ctx)
        print("device MB", used >> 20, flush=True)
        assert used < 800 << 20
        path = [away, away, near, away, near, near]
        outs = [np.empty((h, w, 3), np.uint16) for _ in path]
        for _ in range(2):
            ctx.render_batch(path, outs, out_on_device=False)
            for v, o in zip(path, outs):
                assert np.array_equal(o, a[0] if v is near else away_img)
        p = {"means": means, "log_scales": np.log(scale), "quats": q,
             "opacity_logits": rng.uniform(-4.0, -3.0, n), "sh": rng.uniform(0, 0.5, (n, 1, 3))}
        tr = L.Trainer(ctx, {k: np.ascontiguousarray(v, np.float32) for k, v in p.items()}, 0)
        cfg = L.make_train_cfg()
        first = tr.forward(near, cfg)
        for _ in range(2):
            assert not tr.forward(away, cfg)[0].any()
            assert not tr.forward(away, cfg)[0].any()
            got = tr.forward(near, cfg)
            assert np.array_equal(got[0], first[0]) and np.array_equal(got[1], first[1])
            assert got[3]["pairs_pre"] == first[3]["pairs_pre"] > 1 << 22
    finally:
        ctx.close()
