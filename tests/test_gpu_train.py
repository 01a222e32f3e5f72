"""The HIP training path (gs_train_* entry points) against the reference's own
training dumps (tests/golden/t0_*: fp64 autograd of gsplat/train_oracle.py) and
against the training oracle (oracle/train_oracle.py) on a C5-shaped scene.
Bars: forward values 1e-5 relative, images 1e-4 absolute; gradients rel 1e-2 in
the reference's rel_error (its gate for the device backward); Adam moments
bit-exact, parameters within 1e-7."""
import numpy as np
import pytest

from gsplat_tt_amd import _lib as L
from gsplat_tt_amd import scenes
from oracle import train_oracle as TO
from tests import golden_io
from tests.test_train_oracle import rel_err

pytestmark = pytest.mark.gpu


def _fixture(name):
    g = golden_io.load(name)
    c = g["cfg_json"]
    cfg = L.make_train_cfg(near=c["near"], lowpass=c["lowpass"], alpha_max=c["alpha_max"],
                           alpha_min=c["alpha_min"], t_min=c["t_min"],
                           background=c["background"], lr=g["adam_lr_json"],
                           betas=tuple(g["adam_betas"]), eps=float(g["adam_eps"]))
    view = L.make_view(g["w2c"], g["K"], g["H"], g["W"], tile_size=16)
    params = {k: g["param_" + k].astype(np.float32) for k in TO.PARAM_NAMES}
    return g, cfg, view, params


@pytest.mark.parametrize("name", golden_io.TRAIN_CASES)
def test_train_forward_matches_dump(gpu_ctx, name):
    print("train forward", name, flush=True)
    g, cfg, view, params = _fixture(name)
    tr = L.Trainer(gpu_ctx, params, g["sh_degree"])
    img, T, pj, st = tr.forward(view, cfg, want_proj=True)
    assert np.array_equal(pj["valid"], g["valid"])
    assert np.array_equal(pj["visible"], g["visible"])
    v = g["valid"]
    for k in ("means2d", "conic", "colors", "opacity", "depth"):
        assert np.allclose(pj[k][v], g[k][v], rtol=2e-5, atol=1e-6), k
    assert float(np.abs(img - g["image"]).max()) < 1e-4
    assert float(np.abs(T - g["final_T"]).max()) < 1e-4


@pytest.mark.parametrize("name", golden_io.TRAIN_CASES)
def test_train_backward_matches_dump(gpu_ctx, name):
    print("train backward", name, flush=True)
    g, cfg, view, params = _fixture(name)
    tr = L.Trainer(gpu_ctx, params, g["sh_degree"])
    tr.forward(view, cfg)
    g2d, _ = tr.backward(cfg, dimage=g["dL_dimage"].astype(np.float32), want_g2d=True)
    ref = {"dL_dmeans2d": g2d[:, 0:2], "dL_dconic": g2d[:, 2:5], "dL_dopacity": g2d[:, 5],
           "dL_dcolors": g2d[:, 6:9]}
    for k, a in ref.items():
        e = rel_err(a, g[k])
        print(k, e)
        assert e < 1e-2, k
    grads = tr.read(3)
    for k in TO.PARAM_NAMES:
        e = rel_err(grads[k], g["grad_" + k])
        print("grad", k, e)
        assert e < 1e-2, k


@pytest.mark.parametrize("name", golden_io.TRAIN_CASES)
def test_train_adam_matches_dump(gpu_ctx, name):
    print("train adam", name, flush=True)
    g, cfg, view, params = _fixture(name)
    tr = L.Trainer(gpu_ctx, params, g["sh_degree"])
    tr.write(1, {k: g["adam_m_in_" + k] for k in TO.PARAM_NAMES})
    tr.write(2, {k: g["adam_v_in_" + k] for k in TO.PARAM_NAMES})
    tr.write(3, {k: g["grad_" + k].astype(np.float32) for k in TO.PARAM_NAMES})
    tr.set_visible(g["visible"])
    tr.set_step(int(g["adam_step_in"]))
    tr.adam(cfg)
    p, m, v = tr.read(0), tr.read(1), tr.read(2)
    for k in TO.PARAM_NAMES:
        assert np.array_equal(m[k], g["adam_fp32_m_" + k]), k
        assert np.array_equal(v[k], g["adam_fp32_v_" + k]), k
        assert np.allclose(p[k], g["adam_fp32_param_" + k], rtol=0, atol=1e-7), k



@pytest.mark.parametrize("name", golden_io.TRAIN_CASES)
def test_train_adam_bf16_moments_matches_dump(gpu_ctx, name):
    """k_sparse_adam with bf16-stored moments against the reference's
    moment_dtype=bfloat16 step (train_oracle.py:434-470): moments bit-exact,
    parameters within 1e-7; switching the format carries the moments over."""
    print("train adam bf16 moments", name, flush=True)
    g, cfg, view, params = _fixture(name)
    tr = L.Trainer(gpu_ctx, params, g["sh_degree"])
    try:
        tr.write(1, {k: g["adam_m_in_" + k] for k in TO.PARAM_NAMES})
        tr.set_moments(True)  # fp32 moments carried over, rounded to nearest even
        m_b = tr.read(1)
        for k in TO.PARAM_NAMES:
            assert np.array_equal(m_b[k], TO.bf16_round(g["adam_m_in_" + k])), k
        tr.write(1, {k: g["adam_bf16_m_in_" + k] for k in TO.PARAM_NAMES})
        tr.write(2, {k: g["adam_bf16_v_in_" + k] for k in TO.PARAM_NAMES})
        tr.write(3, {k: g["grad_" + k].astype(np.float32) for k in TO.PARAM_NAMES})
        tr.set_visible(g["visible"])
        tr.set_step(int(g["adam_step_in"]))
        tr.adam(cfg)
        p, m, v = tr.read(0), tr.read(1), tr.read(2)
        for k in TO.PARAM_NAMES:
            assert np.array_equal(m[k], g["adam_bf16_m_" + k]), k
            assert np.array_equal(v[k], g["adam_bf16_v_" + k]), k
            assert np.allclose(p[k], g["adam_bf16_param_" + k], rtol=0, atol=1e-7), k
        tr.set_moments(False)  # back to fp32: the bf16 values exactly
        m32 = tr.read(1)
        for k in TO.PARAM_NAMES:
            assert np.array_equal(m32[k], g["adam_bf16_m_" + k]), k
    finally:
        tr.set_moments(False)

def _c5_small(n=1500, H=90, W=160, seed=55):
    scene, tgt_scene, cams = scenes.config5(seed=seed, n=n)
    K = scenes.intrinsics(0.5 * W / np.tan(np.deg2rad(25.0)), 0.5 * W / np.tan(np.deg2rad(25.0)),
                          W / 2, H / 2)
    return scenes.train_params(scene), scenes.train_params(tgt_scene), cams[0].w2c, K, H, W


def test_train_steps_match_oracle(gpu_ctx):
    """Three whole steps (forward + L1 + backward + sparse Adam) of a C5-shaped
    scene (SH degree 1) against the oracle's steps from the same parameters."""
    print("train steps c5-shaped", flush=True)
    params, tparams, w2c, K, H, W = _c5_small()
    cfg_o = TO.Cfg(sh_degree=1)
    cfg = L.make_train_cfg()
    view = L.make_view(w2c, K, H, W, tile_size=16)
    # target: the oracle's render of the perturbed copy
    _, target, _, _, _ = TO.forward(tparams, w2c, K, H, W, cfg_o)
    target = target.astype(np.float32)
    tr = L.Trainer(gpu_ctx, params, 1)
    p_o = {k: v.astype(np.float32) for k, v in params.items()}
    m_o = {k: np.zeros_like(v) for k, v in p_o.items()}
    v_o = {k: np.zeros_like(v) for k, v in p_o.items()}
    for step in range(3):
        st = tr.step(view, cfg, target)
        pr, img, fT, order, live = TO.forward(p_o, w2c, K, H, W, cfg_o)
        loss, dimg = TO.l1_loss_grad(img, target)
        g2 = TO.blend_backward(pr, order, live, fT, dimg, H, W, cfg_o)
        grads = TO.projection_backward(pr, g2, cfg_o)
        out = TO.sparse_adam(p_o, grads, m_o, v_o, step, pr["visible"])
        p_o = {k: out[k][0] for k in out}
        m_o = {k: out[k][1] for k in out}
        v_o = {k: out[k][2] for k in out}
        print(f"step {step}: loss gpu {st['loss']:.6f} oracle {loss:.6f}, M {st['num_blendable']}"
              f" P {st['num_entries']}")
        assert abs(st["loss"] - loss) <= 1e-4 * max(loss, 1e-6) + 1e-7
    p = tr.read(0)
    for k in TO.PARAM_NAMES:
        d = np.abs(p[k] - p_o[k]).max()
        moved = np.abs(p_o[k] - params[k]).max()
        print(k, "max diff", d, "moved", moved)
        assert d <= 1e-2 * max(moved, 1e-12) + 1e-6, k


@pytest.mark.parametrize("name", golden_io.TRAIN_CASES)
def test_train_loss_ssim_matches_dump(gpu_ctx, name):
    """gs_train_loss with lambda 0.2 is the reference's full loss: its value and
    dL/dimage against the dump (fp64 autograd of 0.8 L1 + 0.2 (1 - SSIM)), on the
    dump's image rounded to fp32 (the oracle re-evaluated on those inputs pins
    the rounding part)."""
    print("train loss ssim", name, flush=True)
    g = golden_io.load(name)
    img, tgt = g["image"].astype(np.float32), g["target"].astype(np.float32)
    loss, l1, ssim, grad = gpu_ctx.train_loss(img, tgt, 0.2)
    lo, l1o, so, go = TO.ssim_loss_grad(img, tgt, 0.2)
    print(f"loss gpu {loss:.9f} oracle {lo:.9f} dump {float(g['loss']):.9f}; "
          f"grad rel {rel_err(grad, go):.3g}")
    assert abs(loss - lo) <= 1e-6 * lo and abs(l1 - l1o) <= 1e-6 * l1o
    assert abs(ssim - so) <= 1e-6
    assert abs(lo - float(g["loss"])) <= 1e-6 * lo  # fp32 rounding of the inputs only
    assert rel_err(grad, go) < 1e-3
    assert rel_err(grad, g["dL_dimage"]) < 1e-2  # the reference's device-backward gate


def test_train_loss_ssim_full_size(gpu_ctx):
    """1280x720 image against a noisy, blurred-edge target: device loss terms and
    gradient against the fp64 oracle; lambda 0 gives the plain L1 gradient."""
    print("train loss ssim 1280x720", flush=True)
    rng = np.random.default_rng(9)
    H, W = 720, 1280
    tgt = rng.uniform(0, 1, (H, W, 3)).astype(np.float32)
    img = np.clip(tgt + rng.normal(0, 0.05, tgt.shape), 0, 1).astype(np.float32)
    img[100:300, 200:600] = 0.5  # a flat patch: low-variance SSIM terms
    loss, l1, ssim, grad = gpu_ctx.train_loss(img, tgt, 0.2)
    lo, l1o, so, go = TO.ssim_loss_grad(img, tgt, 0.2)
    e = rel_err(grad, go)
    print(f"loss gpu {loss:.9f} oracle {lo:.9f} ssim {ssim:.7f}/{so:.7f} grad rel {e:.3g}")
    assert abs(loss - lo) <= 1e-6 * lo and abs(ssim - so) <= 1e-6
    assert e < 1e-3
    l0, l10, s0, g0 = gpu_ctx.train_loss(img, tgt, 0.0, loss_scale=2.0)
    d = img.astype(np.float64) - tgt
    assert s0 == 0.0 and abs(l0 - 2.0 * np.abs(d).mean()) <= 1e-6 * l0
    assert np.array_equal(g0, (np.sign(d) * (2.0 / d.size)).astype(np.float32))


@pytest.mark.parametrize("h,w", [(1, 1), (1, 70), (50, 1), (21, 31), (22, 32), (23, 33), (45, 65)])
def test_train_loss_ssim_tiles(gpu_ctx, h, w):
    """Whole, cut and one-pixel tiles (32 x 22) of the SSIM filters against the fp64
    oracle. Each filter value is 121 fp32 terms of one sign (relative error below
    ~1e-6); the variances in D and B are at least 9e-4, against which the moments'
    error of 1e-6 is 1e-3, the gradient test's bound."""
    print("ssim tiles", h, w, flush=True)
    rng = np.random.default_rng(h + w)
    tgt = rng.uniform(0, 1, (h, w, 3)).astype(np.float32)
    img = np.clip(tgt + rng.normal(0, 0.05, tgt.shape), 0, 1).astype(np.float32)
    loss, l1, ssim, grad = gpu_ctx.train_loss(img, tgt, 0.2)
    lo, l1o, so, go = TO.ssim_loss_grad(img, tgt, 0.2)
    assert abs(loss - lo) <= 1e-6 * lo and abs(ssim - so) <= 1e-6
    assert rel_err(grad, go) < 1e-3


@pytest.mark.parametrize("term", ["A", "B"])
def test_train_loss_ssim_zero_terms(gpu_ctx, term):
    """SSIM = A B / (C D) where A or B passes through 0: pairs of lone pixels, 12 apart, the
    target's stepping through the 400 floats around the one that makes the term 0 (an ulp
    of the term a step, so some step has it exactly 0 in fp32). Loss and gradient are
    finite and the oracle's, whose 64-bit quotients by terms of 1e-12 and more hold to
    1e-8. Bound as in the tiles' test."""
    print("ssim zero terms", term, flush=True)
    g = np.exp(-np.arange(-5, 6) ** 2 / 4.5)
    g2 = (g[5] / g.sum()) ** 2  # the window's middle
    # A = 2 g2^2 a b + c1, B = 2 g2 a b (1 - g2) + c2, with a = 1
    root = -TO.SSIM_C1 / (2 * g2 * g2) if term == "A" else -TO.SSIM_C2 / (2 * g2 * (1 - g2))
    first = np.float32(root).view(np.uint32) - np.uint32(200)
    steps = (first + np.arange(400, dtype=np.uint32)).view(np.float32).reshape(20, 20)
    img, tgt = np.zeros((240, 240, 3), np.float32), np.zeros((240, 240, 3), np.float32)
    img[6::12, 6::12], tgt[6::12, 6::12] = 1.0, steps[..., None]
    loss, l1, ssim, grad = gpu_ctx.train_loss(img, tgt, 0.2)
    lo, l1o, so, go = TO.ssim_loss_grad(img, tgt, 0.2)
    assert np.isfinite(go).all() and np.isfinite(grad).all()
    assert abs(loss - lo) <= 1e-6 * lo and abs(ssim - so) <= 1e-6
    assert rel_err(grad, go) < 1e-3


def test_train_step_ssim_loss_matches_oracle(gpu_ctx):
    """One whole step with the full 3DGS loss (lambda 0.2) of a C5-shaped scene
    against the oracle's forward, SSIM loss gradient, backward and Adam."""
    print("train step ssim c5-shaped", flush=True)
    params, tparams, w2c, K, H, W = _c5_small(seed=57)
    cfg_o = TO.Cfg(sh_degree=1)
    cfg = L.make_train_cfg(lambda_dssim=0.2)
    view = L.make_view(w2c, K, H, W, tile_size=16)
    _, target, _, _, _ = TO.forward(tparams, w2c, K, H, W, cfg_o)
    target = target.astype(np.float32)
    tr = L.Trainer(gpu_ctx, params, 1)
    st = tr.step(view, cfg, target)
    p_o = {k: v.astype(np.float32) for k, v in params.items()}
    pr, img, fT, order, live = TO.forward(p_o, w2c, K, H, W, cfg_o)
    loss, l1, ssim, dimg = TO.ssim_loss_grad(img, target, 0.2)
    g2 = TO.blend_backward(pr, order, live, fT, dimg, H, W, cfg_o)
    grads = TO.projection_backward(pr, g2, cfg_o)
    zeros = {k: np.zeros_like(v) for k, v in p_o.items()}
    out = TO.sparse_adam(p_o, grads, zeros, dict(zeros), 0, pr["visible"])
    print(f"loss gpu {st['loss']:.7f} oracle {loss:.7f}; ssim {st['ssim']:.7f}/{ssim:.7f}")
    assert abs(st["loss"] - loss) <= 1e-4 * loss
    assert abs(st["ssim"] - ssim) <= 1e-5 and abs(st["l1"] - l1) <= 1e-4 * l1
    p = tr.read(0)
    for k in TO.PARAM_NAMES:
        d = np.abs(p[k] - out[k][0]).max()
        moved = np.abs(out[k][0] - params[k]).max()
        print(k, "max diff", d, "moved", moved)
        assert d <= 1e-2 * max(moved, 1e-12) + 1e-6, k



def test_train_pair_capacity_retry():
    """A first training forward whose candidate pairs exceed the context's
    starting capacity (max(2^20, 8N)): 4000 large, faint Gaussians at 320x240
    (300 tiles) give about 1.19M candidates. The forward grows the capacity and
    re-runs: its image and loss equal the oracle's, and its backward equals the
    backward of the same forward run again at the grown capacity (no re-run).
    (The oracle blends every pixel for every Gaussian, so its cost is at least
    256 x 2^20 pixel evaluations: its backward is left to the smaller cases.)"""
    print("train pair-capacity retry", flush=True)
    rng = np.random.default_rng(61)
    n, H, W = 4000, 240, 320
    z = rng.uniform(4.0, 6.0, n)
    params = {
        "means": np.stack([rng.uniform(-1.2, 1.2, n) * z / 4.0,
                           rng.uniform(-0.9, 0.9, n) * z / 4.0, z], -1).astype(np.float32),
        "log_scales": rng.normal(np.log(2.2), 0.1, (n, 3)).astype(np.float32),
        "quats": rng.normal(0, 1, (n, 4)).astype(np.float32),
        "opacity_logits": rng.normal(-3.5, 0.3, n).astype(np.float32),
        "sh": rng.uniform(-0.5, 0.5, (n, 1, 3)).astype(np.float32),
    }
    target = rng.uniform(0.0, 1.0, (H, W, 3)).astype(np.float32)
    w2c = np.eye(4, dtype=np.float32)
    K = scenes.intrinsics(250.0, 250.0, W / 2, H / 2)
    cfg = L.make_train_cfg()
    view = L.make_view(w2c, K, H, W, tile_size=16)
    ctx = L.Context(0)  # a fresh context: the capacity starts at the default
    try:
        tr = L.Trainer(ctx, params, 0)
        img, T, _, st = tr.forward(view, cfg, target)
        print(f"pairs_pre {st['pairs_pre']} capacity {st['pair_capacity']} "
              f"P {st['num_entries']}", flush=True)
        assert st["pairs_pre"] > (1 << 20)
        assert st["pair_capacity"] >= st["pairs_pre"]
        tr.backward(cfg)
        g_retry = tr.read(3)
        cap = st["pair_capacity"]
        img2, _, _, st2 = tr.forward(view, cfg, target)
        assert st2["pair_capacity"] == cap and st2["pairs_pre"] == st["pairs_pre"]
        assert np.array_equal(img2, img) and st2["loss"] == st["loss"]
        tr.backward(cfg)
        g_direct = tr.read(3)
    finally:
        ctx.close()
    for k in TO.PARAM_NAMES:
        # atomics add in another order: equal up to fp32 summation order
        e = rel_err(g_retry[k], g_direct[k])
        d = float(np.abs(g_retry[k] - g_direct[k]).max() / np.abs(g_direct[k]).max())
        print("grad", k, "retry vs direct: rel", e, "max-normalised", d)
        assert e < 1e-2 and d < 1e-4, k
    cfg_o = TO.Cfg(sh_degree=0)
    _, img_o, T_o, _, _ = TO.forward(params, w2c, K, H, W, cfg_o)
    loss_o, _ = TO.l1_loss_grad(img_o, target)
    d = float(np.abs(img - img_o).max())
    print(f"image max_abs {d:.3g}; loss gpu {st['loss']:.7f} oracle {loss_o:.7f}", flush=True)
    assert d < 1e-4 and float(np.abs(T - T_o).max()) < 1e-4
    assert abs(st["loss"] - loss_o) <= 1e-4 * loss_o


@pytest.mark.parametrize("n,H,W,op", [(1, 5, 3, 2.0), (2, 16, 16, 2.0), (63, 23, 40, -2.0),
                                      (64, 16, 32, -2.0), (65, 23, 17, -2.0), (129, 33, 40, -1.0),
                                      (200, 20, 47, 3.0)])
def test_train_bands_match_oracle(gpu_ctx, n, H, W, op):
    """Tile lists around the 64-entry batches of the band kernels and images that cut
    bands and tiles, thin rotated Gaussians among them (the band test must drop only
    what reaches no pixel), sparse to saturated (op = 3: pixels stop early).
    A rounding of alpha may move one entry over the 1/255 threshold at a pixel,
    which changes its colour by at most 1/255 of the entry's (< 1.3): 6e-3; the rest is
    float32 rounding, far below 2e-6 on average. Gradients: the file's bar."""
    print("train bands", n, H, W, op, flush=True)
    rng = np.random.default_rng(1000 + n)
    f = 0.6 * W
    K = scenes.intrinsics(f, f, W / 2, H / 2)
    z = rng.uniform(2, 4, n)
    p = {"means": np.stack([(rng.uniform(-0.1, 1.1, n) - 0.5) * W / f * z,
                            (rng.uniform(-0.1, 1.1, n) - 0.5) * H / f * z, z], 1),
         "log_scales": rng.normal(-2.0, 1.0, (n, 3)), "quats": rng.standard_normal((n, 4)),
         "opacity_logits": rng.normal(op, 1.0, n), "sh": rng.uniform(-0.5, 1.0, (n, 1, 3))}
    p = {k: v.astype(np.float32) for k, v in p.items()}
    bg = (0.3, 0.6, 0.1)
    cfg_o = TO.Cfg(sh_degree=0, background=bg)
    w2c = np.eye(4, dtype=np.float32)
    pr, im, fT, order, live = TO.forward(p, w2c, K, H, W, cfg_o)
    dimg = rng.standard_normal((H, W, 3)).astype(np.float32)
    tr = L.Trainer(gpu_ctx, p, 0)
    cfg = L.make_train_cfg(background=bg)
    img, T, _, _ = tr.forward(L.make_view(w2c, K, H, W, tile_size=16), cfg)
    for a, b in ((img, im), (T, fT)):
        assert float(np.abs(a - b).max()) < 6e-3
        assert float(np.abs(a - b).mean()) < 2e-6
    tr.backward(cfg, dimage=dimg)
    grads = tr.read(3)
    g2 = TO.blend_backward(pr, order, live, fT, dimg.astype(np.float64), H, W, cfg_o)
    ref = TO.projection_backward(pr, g2, cfg_o)
    for k in TO.PARAM_NAMES:
        assert rel_err(grads[k], ref[k]) < 1e-2, k


@pytest.mark.parametrize("n,deg,bf16", [(1, 0, False), (127, 3, False), (129, 2, True),
                                        (255, 1, True), (257, 0, False), (600, 3, True)])
def test_train_step_rows(gpu_ctx, n, deg, bf16):
    """The fused gradient and Adam pass over whole and partial workgroups of rows (128 or
    256), every SH degree (row lengths 14 to 59 values): moments and parameters follow
    bit for bit from the step's own gradients, invisible rows keep theirs, and a row
    whose gradient returns to zero (another view, or gradients written from outside)
    reads zero again."""
    print("train step rows", n, deg, bf16, flush=True)
    rng = np.random.default_rng(n + deg)
    H, W = 40, 56
    K = scenes.intrinsics(60.0, 60.0, W / 2, H / 2)
    side = np.where(rng.random(n) < 0.3, -1.0, 1.0)  # a third behind the camera
    if n == 1:
        side[:] = 1.0
    p = {"means": np.stack([rng.uniform(-0.6, 0.6, n), rng.uniform(-0.4, 0.4, n),
                            side * rng.uniform(2, 4, n)], 1),
         "log_scales": rng.normal(-2.5, 0.5, (n, 3)), "quats": rng.standard_normal((n, 4)),
         "opacity_logits": rng.normal(0, 1.0, n),
         "sh": rng.uniform(-0.5, 0.5, (n, (deg + 1) ** 2, 3))}
    p = {k: v.astype(np.float32) for k, v in p.items()}
    cfg = L.make_train_cfg()
    view = L.make_view(np.eye(4, dtype=np.float32), K, H, W, tile_size=16)
    away = L.make_view(np.diag([1, 1, 1, 1]).astype(np.float32) +
                       np.array([[0, 0, 0, 0], [0, 0, 0, 0], [0, 0, 0, -50], [0, 0, 0, 0]],
                                np.float32), K, H, W, tile_size=16)
    target = rng.random((H, W, 3)).astype(np.float32)
    tr = L.Trainer(gpu_ctx, p, deg)
    try:
        tr.set_moments(bf16)
        _, _, proj, _ = tr.forward(view, cfg, want_proj=True)
        vis = proj["visible"]
        tr.step(view, cfg, target)
        g, m, v, q = tr.read(3), tr.read(1), tr.read(2), tr.read(0)
        f = np.float32
        rnd = TO.bf16_round if bf16 else (lambda x: x)
        bc1, bc2 = 1.0 - 0.9, 1.0 - 0.999
        lr = {"means": cfg.lr_means, "log_scales": cfg.lr_log_scales, "quats": cfg.lr_quats,
              "opacity_logits": cfg.lr_opacity}
        for k in TO.PARAM_NAMES:
            assert np.abs(g[k]).max() > 0, k
            m1, v1 = f(1.0 - 0.9) * g[k], f(1.0 - 0.999) * g[k] * g[k]
            den = np.sqrt(v1) / f(np.sqrt(bc2)) + f(cfg.eps)
            if k == "sh":
                step = np.full((1, (deg + 1) ** 2, 1), f(cfg.lr_sh_rest) / f(bc1), f)
                step[:, 0] = f(cfg.lr_sh_dc) / f(bc1)
            else:
                step = f(lr[k] / bc1)
            row = vis.reshape(-1, *([1] * (g[k].ndim - 1)))
            assert np.array_equal(m[k], np.where(row, rnd(m1), f(0))), k
            assert np.array_equal(v[k], np.where(row, rnd(v1), f(0))), k
            assert np.array_equal(q[k], np.where(row, p[k] - step * (m1 / den), p[k])), k
        tr.step(away, cfg, target)  # nothing in view: every gradient is zero again
        assert all(np.all(a == 0) for a in tr.read(3).values())
        after = tr.read(0)
        assert all(np.array_equal(after[k], q[k]) for k in TO.PARAM_NAMES)
        tr.write(3, {k: np.ones_like(a) for k, a in g.items()})
        tr.forward(away, cfg, target)
        tr.backward(cfg)
        assert all(np.all(a == 0) for a in tr.read(3).values())
    finally:
        tr.set_moments(False)


def test_train_step_capacity_rerun():
    """A first step whose candidate pairs exceed the starting capacity (2000 Gaussians over
    most of 3600 tiles) is run again whole: the attempt that did not fit leaves
    parameters, moments and the step count alone, so one Adam step has been taken."""
    print("train step capacity", flush=True)
    rng = np.random.default_rng(4)
    n, H, W = 2000, 720, 1280
    p = {"means": np.stack([rng.uniform(-1, 1, n), rng.uniform(-1, 1, n),
                            rng.uniform(3, 5, n)], 1),
         "log_scales": rng.normal(0.3, 0.1, (n, 3)), "quats": rng.standard_normal((n, 4)),
         "opacity_logits": rng.normal(-3, 0.3, n), "sh": rng.uniform(-0.5, 0.5, (n, 1, 3))}
    p = {k: v.astype(np.float32) for k, v in p.items()}
    K = scenes.intrinsics(1000.0, 1000.0, W / 2, H / 2)
    view = L.make_view(np.eye(4, dtype=np.float32), K, H, W, tile_size=16)
    ctx = L.Context(0)
    try:
        tr = L.Trainer(ctx, p, 0)
        st = tr.step(view, L.make_train_cfg(), np.zeros((H, W, 3), np.float32))
        assert st["pairs_pre"] > (1 << 20) and st["step"] == 1, st
        assert st["pair_capacity"] >= st["pairs_pre"]
        g, m = tr.read(3), tr.read(1)
        for k in TO.PARAM_NAMES:
            assert np.array_equal(m[k], np.float32(1.0 - 0.9) * g[k]), k
    finally:
        ctx.close()


@pytest.mark.parametrize("n,deg", [(1, 0), (3, 3), (5001, 2), (35_544, 3), (35_545, 3),
                                   (95_000, 3), (91_181, 1)])
def test_train_arrays_round_trip(gpu_ctx, n, deg):
    """Parameters, moments (fp32 and bf16) and gradients come back as they were written:
    one chunk of the staged transfer, its edge (35544 rows of degree 3 fill 8 MiB), several."""
    print("train arrays", n, deg, flush=True)
    rng = np.random.default_rng(n)
    shp = {"means": (n, 3), "log_scales": (n, 3), "quats": (n, 4), "opacity_logits": (n,),
           "sh": (n, (deg + 1) ** 2, 3)}
    arrs = [{k: rng.standard_normal(s, dtype=np.float32) for k, s in shp.items()}
            for _ in range(4)]
    tr = L.Trainer(gpu_ctx, arrs[0], deg)
    try:
        for which in (1, 2, 3):
            tr.write(which, arrs[which])
        for which in range(4):
            got = tr.read(which)
            assert all(np.array_equal(got[k], arrs[which][k]) for k in shp), which
        tr.set_moments(True)
        got = tr.read(2)
        assert all(np.array_equal(got[k], TO.bf16_round(arrs[2][k])) for k in shp)
        tr.write(1, arrs[3])
        got = tr.read(1)
        assert all(np.array_equal(got[k], TO.bf16_round(arrs[3][k])) for k in shp)
        got = tr.read(0)
        assert all(np.array_equal(got[k], arrs[0][k]) for k in shp)
    finally:
        tr.set_moments(False)


def _spread_params(rng, n, W, H, f):
    z = rng.uniform(2, 4, n)
    p = {"means": np.stack([rng.uniform(-0.5, 0.5, n) * W / f * z,
                            rng.uniform(-0.5, 0.5, n) * H / f * z, z], 1),
         "log_scales": rng.normal(np.log(18.0 / f), 0.3, (n, 3)),  # about 6 pixels
         "quats": rng.standard_normal((n, 4)), "opacity_logits": rng.normal(0, 1.0, n),
         "sh": rng.uniform(-0.5, 0.5, (n, 1, 3))}
    return {k: v.astype(np.float32) for k, v in p.items()}


@pytest.mark.parametrize("h,w", [(40, 56), (129 * 16, 128 * 16 + 1), (32, 33_000 * 16)])
def test_train_backward_after_a_sort(h, w):
    """A standalone sort between a forward and its backward (binned; by blocks, two sort
    passes; sorted by tile, three) leaves the forward's ids, records and ranges alone:
    the gradients are those of a backward right after the forward, but for the order
    of the atomic adds: float32 sums of some 50 band terms, 50 x 2^-24 = 3e-6 of the
    terms' magnitude, of which a mean's gradient keeps a tenth or more in the 2-norm
    (single elements may cancel to nothing, so not element by element): 1e-4."""
    print("train sort between", h, w, flush=True)
    rng = np.random.default_rng(h)
    f = 0.9 * w
    p = _spread_params(rng, 3000, w, h, f)
    view = L.make_view(np.eye(4, dtype=np.float32), scenes.intrinsics(f, f, w / 2, h / 2), h, w,
                       tile_size=16)
    cfg = L.make_train_cfg()
    target = np.zeros((h, w, 3), np.float32)
    n, tiles = 100_003, 500
    keys = (rng.integers(0, tiles, n).astype(np.uint64) << np.uint64(32)) | \
        rng.uniform(1, 2, n).astype(np.float32).view(np.uint32).astype(np.uint64)
    ctx = L.Context(0)
    ptrs = []
    try:
        tr = L.Trainer(ctx, p, 0)
        tr.forward(view, cfg, target)
        tr.backward(cfg)
        ref = tr.read(3)
        ptrs = [ctx.dev_alloc(8 * n), ctx.dev_alloc(4 * n), ctx.dev_alloc(8 * tiles)]
        for ids in (False, True):
            tr.forward(view, cfg, target)
            ctx.h2d(ptrs[0], keys)
            ctx.h2d(ptrs[1], np.arange(n, dtype=np.uint32))
            sort = ctx.sort_tile_depth_ids_dev if ids else ctx.sort_tile_depth_dev
            sort(ptrs[0], ptrs[1], n, tiles, ptrs[2])
            tr.backward(cfg)
            got = tr.read(3)
            for k in TO.PARAM_NAMES:
                assert np.abs(ref[k]).max() > 0, k
                assert np.linalg.norm(got[k] - ref[k]) < 1e-4 * np.linalg.norm(ref[k]), (k, ids)
    finally:
        for q in ptrs:
            ctx.dev_free(q)
        ctx.close()


def test_train_backward_needs_its_buffers(gpu_ctx):
    """Calls that overwrite what a forward left (projection, tile assignment, binning,
    blending, a loss, a frame) make its backward an error; with nothing to do they
    leave it."""
    print("train buffers", flush=True)
    rng = np.random.default_rng(2)
    h, w, n = 40, 56, 200
    p = _spread_params(rng, n, w, h, 50.0)
    view = L.make_view(np.eye(4, dtype=np.float32), scenes.intrinsics(50.0, 50.0, w / 2, h / 2),
                       h, w, tile_size=16, output="f32")
    cfg = L.make_train_cfg()
    cov = scenes.cov3d(np.exp(p["log_scales"]), p["quats"] /
                       np.linalg.norm(p["quats"], axis=1, keepdims=True))
    op, col = np.full(n, 0.5, np.float32), rng.random((n, 3)).astype(np.float32)
    pr = gpu_ctx.project(p["means"], cov, op, col, view)
    assign = (pr["means2d"], pr["radii"], h, w, 16, pr["covs2d"], pr["opacities"])
    g, t, _ = gpu_ctx.tile_assign(*assign)
    ids, ranges = gpu_ctx.sort_and_bin(g, t, pr["depths"], 4, 3)
    img = np.zeros((h, w, 3), np.float32)
    calls = {
        "project": lambda: gpu_ctx.project(p["means"], cov, op, col, view),
        "tile_assign": lambda: gpu_ctx.tile_assign(*assign),
        "sort_and_bin": lambda: gpu_ctx.sort_and_bin(g, t, pr["depths"], 4, 3),
        "cull_and_blend": lambda: gpu_ctx.cull_and_blend(
            pr["means2d"], pr["covs2d"], pr["colors"], pr["opacities"], ids, ranges, view),
        "loss": lambda: gpu_ctx.train_loss(img, img + 0.5, 0.2),
        "render": lambda: (gpu_ctx.set_scene(p["means"], cov, op, col), gpu_ctx.render(view)),
    }
    tr = L.Trainer(gpu_ctx, p, 0)
    for name, call in calls.items():
        tr.forward(view, cfg, img)
        call()
        with pytest.raises(ValueError, match="no current forward"):
            tr.backward(cfg)
    tr.forward(view, cfg, img)
    gpu_ctx.tile_assign(*(a[:0] for a in assign[:2]), h, w, 16)
    gpu_ctx.sort_and_bin(g[:0], t[:0], pr["depths"], 4, 3)
    tr.backward(cfg)
    assert any(np.abs(a).max() > 0 for a in tr.read(3).values())


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_train_nonfinite_colour_stays_where_it_blends(gpu_ctx, bad):
    """A Gaussian with a non-finite colour changes only the pixels that blend it, as
    when a skipped or unreached entry is not read (train_oracle.py:213-229): those
    are found with two finite colours. Behind three opaque Gaussians it blends
    nowhere; beside unrelated pixels of the same 16 x 4 bands it blends its own few. The
    image elsewhere is the same bit for bit, and so are the other Gaussians' gradients
    from those pixels but for the order of the atomic adds (50 x 2^-24 of the terms,
    a tenth of which is left: 1e-4)."""
    print("train nonfinite", bad, flush=True)
    h, w, f = 33, 48, 40.0
    view = L.make_view(np.eye(4, dtype=np.float32), scenes.intrinsics(f, f, w / 2, h / 2), h, w,
                       tile_size=16)
    cfg = L.make_train_cfg(background=(0.2, 0.4, 0.6))
    rng = np.random.default_rng(9)
    dimage = rng.standard_normal((h, w, 3)).astype(np.float32)

    def gaussian(px, py, z, size, logit):
        return [(px - w / 2) / f * z, (py - h / 2) / f * z, z], np.log(size * z / f), logit

    wall = [gaussian(w / 2, h / 2, 1.0 + 0.1 * k, 400.0, 9.0) for k in range(3)]
    small = [gaussian(x, y, 3.0, 0.7, 1.0) for x in (3, 9, 21, 30, 44) for y in (3, 6, 9, 18, 27)]
    hidden, beside = gaussian(w / 2, h / 2, 5.0, 6.0, 2.0), gaussian(14.5, 6.5, 4.0, 0.7, 2.0)
    for name, rows in (("hidden", wall + small + [hidden]), ("beside", small + [beside])):
        n = len(rows)
        p = {"means": np.array([r[0] for r in rows]),
             "log_scales": np.array([[r[1]] * 3 for r in rows]) + rng.normal(0, 0.05, (n, 3)),
             "quats": rng.standard_normal((n, 4)),
             "opacity_logits": np.array([r[2] for r in rows]),
             "sh": rng.uniform(0.2, 1.0, (n, 1, 3))}
        p = {k: np.ascontiguousarray(v, np.float32) for k, v in p.items()}

        def forward(colour):
            q = {k: v.copy() for k, v in p.items()}
            q["sh"][-1] = colour
            tr = L.Trainer(gpu_ctx, q, 0)
            return (tr,) + tr.forward(view, cfg)[:2]

        def gradients(tr, pixels):
            tr.backward(cfg, dimage=np.where(pixels[..., None], dimage, np.float32(0)))
            return tr.read(3)

        img0 = forward(0.3)[1]
        tr, img1, T1 = forward(40.0)
        clean = (img0 == img1).all(2)  # pixels that do not blend it
        assert clean.all() if name == "hidden" else (~clean).any() and clean.sum() > h * w // 2
        ref = gradients(tr, clean)
        tr, img, T = forward(bad)
        assert np.array_equal(img[clean], img0[clean]), name
        assert np.array_equal(T, T1), name
        got = gradients(tr, clean)
        for k in TO.PARAM_NAMES:
            a, b = got[k][:-1], ref[k][:-1]
            assert np.isfinite(a).all(), (name, k)
            assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b), (name, k)
            if name == "hidden":
                assert not got[k][-1].any(), k


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_train_nonfinite_pixel_gradient_stays_where_it_blends(gpu_ctx, bad):
    """A non-finite gradient of one pixel reaches the Gaussians that this pixel blends and
    no other: not those that only other pixels of the band blend, nor what is summed
    beside them (the entries go in twos, an odd last one with padding that carries the
    id 0). The others' gradients are those with that pixel's gradient at 0, but for the
    order of the atomic adds (20 x 2^-24 of the terms, a tenth of which is left: 1e-4)."""
    print("train nonfinite pixel", bad, flush=True)
    h, w, f = 33, 48, 40.0
    view = L.make_view(np.eye(4, dtype=np.float32), scenes.intrinsics(f, f, w / 2, h / 2), h, w,
                       tile_size=16)
    cfg = L.make_train_cfg(background=(0.2, 0.4, 0.6))
    rng = np.random.default_rng(11)
    dimage = rng.standard_normal((h, w, 3)).astype(np.float32)
    for count in (2, 3, 4, 5):  # entries of the pixel's band, even and odd
        # the first far from the band, then a column of one pixel's width in it
        at = [(40.5, 28.5)] + [(4.5 + 2.5 * k, 9.5) for k in range(count)]
        z = 3.0 + 0.25 * np.arange(len(at))
        p = {"means": np.stack([(np.array([a[0] for a in at]) - w / 2) / f * z,
                                (np.array([a[1] for a in at]) - h / 2) / f * z, z], 1),
             "log_scales": np.log(0.3 * z / f)[:, None].repeat(3, 1) +
             rng.normal(0, 0.05, (len(at), 3)),
             "quats": rng.standard_normal((len(at), 4)), "opacity_logits": np.full(len(at), 1.0),
             "sh": rng.uniform(0.2, 1.0, (len(at), 1, 3))}
        p = {k: np.ascontiguousarray(v, np.float32) for k, v in p.items()}
        tr = L.Trainer(gpu_ctx, p, 0)

        def gradients(value):
            tr.forward(view, cfg)
            d = dimage.copy()
            d[9, 4] = value
            tr.backward(cfg, dimage=d)
            return tr.read(3)

        ref, got = gradients(0.0), gradients(bad)
        assert not np.isfinite(got["sh"][1]).any()  # the pixel blends it
        others = [0] + list(range(3, len(at)))  # 5 pixels and more from it
        for k in TO.PARAM_NAMES:
            a, b = got[k][others], ref[k][others]
            assert np.isfinite(a).all(), (count, k)
            assert np.abs(b[0]).max() > 0 or k == "quats", (count, k)
            assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b), (count, k)
