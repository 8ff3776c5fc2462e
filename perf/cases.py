"""The work that users of this package have it do, as measurable cases.

    listed()            the named cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs on the GPU, and what a program keeps between calls
    run(state)          one pass through the public entry points, and its outputs
    work(case)          the bytes and operations a pass cannot do without
    tolerance(case)     how far a correct implementation's outputs may be off
    exact(case, seed)   the outputs in 64 bits, in plain torch

Kinds of case:

    view    one differentiable 3D view: amdsplat.rasterize and its backward (the training path)
    infer   one 3D view without gradients: amdsplat.rasterize_inference (evaluation, viewers)
    step    a whole training step: rasterize, l1_ssim_loss, backward, FusedAdam
    loss    l1_ssim_loss and its image gradient on a frame
    adam    FusedAdam.step over the six parameter groups of a model
    fit     the 2D image-fit step: activation, binning, gs2d.rasterize, squared error, gradients
    toy2d   gs2d.bin_gaussians, gs2d.rasterize and its backward on given 2D Gaussians
    phase0  splat2d.render and its backward
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "3dgs-project_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda"
TILE = 16
LEARNING_RATES = {"means": 1.6e-4, "scales": 5e-3, "quats": 1e-3, "sh_dc": 2.5e-3, "sh_rest": 1.25e-4,
                  "opacity": 5e-2}


def listed():
    return [
        # the smallest call in use: the smoke scene of a unit test or a notebook; launches and host
        # work are all of it
        dict(name="view_2k", kind="view", n=2000, width=160, height=120, degree=3, split=False, antialias=False,
             stats=0, scene="front"),
        # 100k Gaussians without view-dependent colour at 800x800 (an object scene early in training)
        dict(name="view_100k_sh0", kind="view", n=100_000, width=800, height=800, degree=0, split=False,
             antialias=False, stats=0, scene="object"),
        # a mid-size training view with what trainers switch on: the DC / rest pair, antialiasing and
        # densification statistics with absolute gradients, at an odd frame size
        dict(name="view_300k_options", kind="view", n=300_007, width=1001, height=667, degree=2, split=True,
             antialias=True, stats=3, scene="orbit"),
        # the benchmark's view: 1M Gaussians, SH degree 3, 1297x840
        dict(name="view_1m_sh3", kind="view", n=1_000_000, width=1297, height=840, degree=3, split=False,
             antialias=False, stats=0, scene="orbit"),
        # the largest: 3M Gaussians, SH degree 3, 1957x1091, long tile lists
        dict(name="view_3m_sh3", kind="view", n=3_000_000, width=1957, height=1091, degree=3, split=False,
             antialias=False, stats=0, scene="orbit_dense"),
        # rendering a trained model for evaluation or a viewer
        dict(name="infer_1m_sh3", kind="infer", n=1_000_000, width=1297, height=840, degree=3, split=True,
             antialias=False, scene="orbit"),
        # a whole training step with the visibility-masked optimizer
        dict(name="step_100k_sh3", kind="step", n=100_000, width=800, height=800, degree=3, masked=True,
             scene="object"),
        # the training loss alone, on the benchmark's frame
        dict(name="loss_840x1297", kind="loss", channels=3, width=1297, height=840, lam=0.2),
        # the optimizer alone: 59 parameters of 1M Gaussians, float32 moments
        dict(name="adam_1m", kind="adam", n=1_000_000, degree=3, visible=1.0, lowp=False),
        # the 2D image fit: 4096 Gaussians on 256x256
        dict(name="fit_4k_256", kind="fit", n=4096, width=256, height=256),
        # the largest of the 2D benchmark's scenes
        dict(name="toy2d_200k_1024", kind="toy2d", n=200_000, width=1024, height=1024, backend="splat"),
        # the full-HD 2D benchmark scene
        dict(name="phase0_50k_1080p", kind="phase0", n=50_000, width=1920, height=1080, mode="splat", f64=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["view", "view", "view", "infer", "step", "loss", "adam", "fit", "toy2d", "phase0"])
    if kind in ("view", "infer", "step"):
        n = _log_int(rng, 2000, 1_500_000)
        top = 1.0 if n > 50_000 else 0.5
        c = dict(kind=kind, n=n, width=_log_int(rng, 160, 1960 * top), height=_log_int(rng, 120, 1100 * top),
                 degree=rng.choice([0, 1, 2, 3, 3]), scene="object" if n < 200_000 else "orbit")
        if kind == "step":
            c.update(masked=rng.random() < 0.5)
        else:
            c.update(split=rng.random() < 0.5, antialias=rng.random() < 0.3)
        if kind == "view":
            c.update(stats=rng.choice([0, 0, 2, 3]))
        return c
    if kind == "loss":
        return dict(kind=kind, channels=rng.choice([1, 3, 3, 3]), width=_log_int(rng, 60, 1960),
                    height=_log_int(rng, 60, 1100), lam=rng.choice([0.2, 0.2, 1.0]))
    if kind == "adam":
        return dict(kind=kind, n=_log_int(rng, 2000, 2_000_000), degree=rng.choice([0, 1, 2, 3, 3]),
                    visible=rng.choice([1.0, 1.0, 0.7, 0.4]), lowp=rng.random() < 0.25)
    if kind == "fit":
        return dict(kind=kind, n=_log_int(rng, 500, 60_000), width=_log_int(rng, 100, 800),
                    height=_log_int(rng, 100, 800))
    if kind == "toy2d":
        return dict(kind=kind, n=_log_int(rng, 10_000, 200_000), width=_log_int(rng, 256, 1024),
                    height=_log_int(rng, 256, 1024), backend=rng.choice(["splat", "splat", "pixel"]))
    # (the per-pixel backward and float64 cost several times as much per splat)
    mode, f64 = rng.choice(["splat", "splat", "splat", "pixel"]), rng.random() < 0.25
    top = 100_000 if mode == "splat" and not f64 else 10_000
    return dict(kind=kind, n=_log_int(rng, 1000, top), width=_log_int(rng, 200, 1920),
                height=_log_int(rng, 200, 1080), mode=mode, f64=f64)


# ---- inputs -----------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 13)


def _u(g, lo, hi, *shape, dtype=torch.float32):
    return lo + (hi - lo) * torch.rand(*shape, generator=g, device=DEV, dtype=dtype)


def _model(case, g):
    """Raw parameters of n Gaussians: means, log-scales, quaternions, opacity logits, SH [n, K, 3]."""
    n, K, scene = case["n"], (case["degree"] + 1) ** 2, case["scene"]

    def randn(*s):
        return torch.randn(*s, generator=g, device=DEV)

    if scene == "front":  # in front of an identity camera, slightly beyond the frustum, larger splats
        w, h = case["width"], case["height"]
        z = _u(g, 2.0, 8.0, n)
        f = 0.9 * w
        means = torch.stack([_u(g, -0.6, 0.6, n) * w / f * z, _u(g, -0.6, 0.6, n) * h / f * z, z], -1)
        log_scales = torch.log(_u(g, 0.01, 0.1, n, 3))
        o = _u(g, 0.05, 0.95, n)
        logits = torch.log(o / (1.0 - o))
    elif scene == "object":  # a ball of Gaussians seen from outside
        means = 0.5 * randn(n, 3)
        log_scales = _u(g, -5.0, -2.0, n, 3)
        logits = randn(n)
    else:  # 80% in a ball that the camera stands near, 20% in a far shell
        ball = int(round(0.8 * n))
        d = randn(n - ball, 3)
        shell = d / d.norm(dim=1, keepdim=True) * _u(g, 8.0, 12.0, n - ball, 1)
        means = torch.cat([randn(ball, 3), shell], 0)
        mu, sigma = (-4.0, 1.2) if scene == "orbit_dense" else (-4.5, 1.0)
        log_scales = mu + sigma * randn(n, 3)
        logits = -1.0 + 1.5 * randn(n)
    quats = randn(n, 4)
    quats = quats / quats.norm(dim=1, keepdim=True)
    sh = torch.empty(n, K, 3, device=DEV)
    sh[:, 0] = 0.5 * randn(n, 3)
    if K > 1:
        sh[:, 1:] = 0.05 * randn(n, K - 1, 3)
    return means.contiguous(), log_scales.contiguous(), quats.contiguous(), logits.contiguous(), sh


def _camera(case, seed):
    """(viewmat [4, 4], K [3, 3], near, far) on the host, as programs hold them."""
    w, h, scene = case["width"], case["height"], case["scene"]
    g = torch.Generator().manual_seed(int(seed) + 101)
    r = torch.rand(3, generator=g).tolist()
    if scene == "front":
        f, near, far = 0.9 * w, 0.2, 1000.0
        vm = torch.eye(4)
        return vm, torch.tensor([[f, 0.0, w / 2 + 0.3], [0.0, f, h / 2 - 0.2], [0.0, 0.0, 1.0]]), near, far
    near, far = 0.01, 100.0
    if scene == "object":
        f, radius = 1.389 * max(w, h), 4.0
    else:
        f, radius = (0.741 if scene == "orbit_dense" else 0.894) * w, 3.0 + 2.0 * r[0]
    az, el = 2.0 * math.pi * r[1], r[2] - 0.5
    eye = torch.tensor([radius * math.cos(el) * math.cos(az), radius * math.cos(el) * math.sin(az),
                        radius * math.sin(el)], dtype=torch.float64)
    fwd = -eye / eye.norm()
    right = torch.linalg.cross(fwd, torch.tensor([0.0, 0.0, 1.0], dtype=torch.float64))
    right = right / right.norm()
    R = torch.stack([right, torch.linalg.cross(fwd, right), fwd])
    vm = torch.eye(4, dtype=torch.float64)
    vm[:3, :3] = R
    vm[:3, 3] = -R @ eye
    return vm.float(), torch.tensor([[f, 0.0, w / 2.0], [0.0, f, h / 2.0], [0.0, 0.0, 1.0]]), near, far


def _view_inputs(case, seed):
    g = _gen(seed)
    model = _model(case, g)
    vm, K, near, far = _camera(case, seed)
    return g, model, dict(viewmat=vm, K=K, W=case["width"], H=case["height"], near=near, far=far)


def _moments(g, p):
    """Adam moments as they stand some way into training."""
    m = 1e-4 * torch.randn(p.shape, generator=g, device=DEV)
    v = 1e-8 * (0.5 + torch.rand(p.shape, generator=g, device=DEV))
    return m, v


def _optimizer(params, g, sparse, lowp=False):
    from amdsplat import FusedAdam

    groups = [{"params": [p], "lr": LEARNING_RATES[k], "name": k} for k, p in params.items()]
    opt = FusedAdam(groups, lr=0.0, eps=1e-15, sparse=sparse, lowp_moment_groups=("sh_rest",) if lowp else ())
    for k, p in params.items():
        m, v = _moments(g, p)
        if lowp and k == "sh_rest":
            m, v = m.bfloat16(), v.bfloat16()
        opt.state[p] = {"step": 100, "exp_avg": m, "exp_avg_sq": v}
    return opt


def _split_params(model):
    m, ls, q, op, sh = model
    return {"means": m, "scales": ls, "quats": q, "sh_dc": sh[:, :1].contiguous(), "sh_rest": sh[:, 1:].contiguous(),
            "opacity": op}


def _gaussians2d(case, seed):
    """Raw parameters of the 2D models: positions, log-scales, angles, colour and opacity logits, depth."""
    n, w, h = case["n"], case["width"], case["height"]
    g = _gen(seed)
    xy = torch.rand(n, 2, generator=g, device=DEV) * torch.tensor([float(w), float(h)], device=DEV)
    if case["kind"] == "fit":
        log_scale = math.log(2.0) + 0.3 * torch.randn(n, 2, generator=g, device=DEV)
    else:
        log_scale = torch.log(0.5 * math.sqrt(h * w / n) * _u(g, 0.5, 1.5, n, 2))
    theta = _u(g, 0.0, math.pi, n)
    rgb = 0.5 * torch.randn(n, 3, generator=g, device=DEV)
    logit = 0.5 * torch.randn(n, generator=g, device=DEV)
    depth = torch.rand(n, generator=g, device=DEV)
    return g, xy, log_scale, theta, rgb, logit, depth


def _phase0_inputs(case, seed):
    """means, Cholesky factors (sigma 2-10 px), opacity logits, colours, upstream gradient."""
    n, w, h = case["n"], case["width"], case["height"]
    g, f = _gen(seed), torch.float64
    means = torch.stack([_u(g, -0.02 * w, 1.02 * w, n, dtype=f), _u(g, -0.02 * h, 1.02 * h, n, dtype=f)], -1)
    l0, l2 = 1.0 / _u(g, 2.0, 10.0, n, dtype=f), 1.0 / _u(g, 2.0, 10.0, n, dtype=f)
    l1 = _u(g, -0.5, 0.5, n, dtype=f) * torch.minimum(l0, l2)
    o = _u(g, 0.05, 0.6, n, dtype=f)
    got = [means, torch.stack([l0, l1, l2], -1), torch.log(o / (1.0 - o)), torch.rand(n, 3, generator=g, device=DEV,
                                                                                       dtype=f),
           torch.randn(h, w, 3, generator=g, device=DEV, dtype=f)]
    return [t.to(f if case["f64"] else torch.float32).contiguous() for t in got]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("view", "infer"):
        g, model, cam = _view_inputs(case, seed)
        m, ls, q, op, sh = model
        sh = (sh[:, :1].contiguous(), sh[:, 1:].contiguous()) if case["split"] else sh
        opts = dict(cam, proper_antialiasing=case["antialias"], bg=(0.1, 0.2, 0.3))
        state = dict(case=case, opts=opts)
        if kind == "infer":
            return dict(state, params=(m, ls, q, op, sh))
        leaves = [t.requires_grad_(True) for t in (m, ls, q, op, *(sh if case["split"] else (sh,)))]
        grad = torch.randn(3, case["height"], case["width"], generator=g, device=DEV)
        return dict(state, leaves=leaves, grad=grad)
    if kind == "step":
        g, model, cam = _view_inputs(case, seed)
        params = {k: torch.nn.Parameter(v) for k, v in _split_params(model).items()}
        target = torch.rand(3, case["height"], case["width"], generator=g, device=DEV)
        return dict(case=case, opts=cam, params=params, target=target,
                    opt=_optimizer(params, g, sparse=case["masked"]))
    if kind == "loss":
        g = _gen(seed)
        shape = (case["channels"], case["height"], case["width"])
        target = torch.rand(shape, generator=g, device=DEV)
        image = (target + 0.1 * torch.randn(shape, generator=g, device=DEV)).clamp(0.0, 1.0).requires_grad_(True)
        return dict(case=case, image=image, target=target)
    if kind == "adam":
        g = _gen(seed)
        params = {k: torch.nn.Parameter(v) for k, v in _split_params(_model(dict(case, scene="orbit"), g)).items()}
        opt = _optimizer(params, g, sparse=case["visible"] < 1.0, lowp=case["lowp"])
        for p in params.values():
            p.grad = 1e-4 * torch.randn(p.shape, generator=g, device=DEV)
        vis = None
        if case["visible"] < 1.0:
            vis = (torch.rand(case["n"], generator=g, device=DEV) < case["visible"]).to(torch.int32)
        return dict(case=case, params=params, opt=opt, visibility=vis)
    if kind == "fit":
        from gs2d import Gaussians2D

        g, xy, log_scale, theta, rgb, logit, depth = _gaussians2d(case, seed)
        model = Gaussians2D(case["n"], case["height"], case["width"]).to(DEV)
        with torch.no_grad():
            for p, v in ((model.xy, xy), (model.log_scale, log_scale), (model.theta, theta), (model.rgb_logit, rgb),
                         (model.opacity_logit, logit), (model.depth, depth)):
                p.copy_(v)
        return dict(case=case, model=model, target=torch.rand(3, case["height"], case["width"], generator=g,
                                                              device=DEV))
    if kind == "toy2d":
        from gs2d.params import activate, radii_from_cov

        g, xy, log_scale, theta, rgb, logit, depth = _gaussians2d(case, seed)
        means, conic, color, opacity, cov = activate(xy, log_scale, theta, rgb, logit)
        grad = torch.randn(3, case["height"], case["width"], generator=g, device=DEV)
        return dict(case=case, leaves=[t.contiguous().requires_grad_(True) for t in (means, conic, color, opacity)],
                    radii=radii_from_cov(cov), depth=depth, grad=grad)
    *params, grad = _phase0_inputs(case, seed)
    return dict(case=case, leaves=[t.requires_grad_(True) for t in params], grad=grad)


# ---- one pass ---------------------------------------------------------------------------------


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "view":
        from amdsplat import rasterize

        m, ls, q, op, *sh = state["leaves"]
        info = torch.zeros(case["stats"], case["n"], device=DEV) if case["stats"] else None
        image, alpha, aux = rasterize(m, ls, q, op, tuple(sh) if case["split"] else sh[0], densification_info=info,
                                      **state["opts"])
        grads = torch.autograd.grad(image, state["leaves"], state["grad"])
        return {"image": image, "alpha": alpha, "touched": aux["tiles_touched"], "grads": list(grads),
                "stats": list(info) if case["stats"] else None}
    if kind == "infer":
        from amdsplat import rasterize_inference

        return list(rasterize_inference(*state["params"], **state["opts"]))
    if kind == "step":
        from amdsplat import l1_ssim_loss, rasterize

        p, opt = state["params"], state["opt"]
        image, _, aux = rasterize(p["means"], p["scales"], p["quats"], p["opacity"], (p["sh_dc"], p["sh_rest"]),
                                  **state["opts"])
        loss = l1_ssim_loss(image, state["target"], 0.2)
        loss.backward()
        opt.step(visibility=aux["visibility"] if case["masked"] else None)
        opt.zero_grad(set_to_none=True)
        return {"image": image, "loss": loss, "params": [t.detach() for t in p.values()],
                "m": [opt.state[t]["exp_avg"] for t in p.values()]}
    if kind == "loss":
        from amdsplat import l1_ssim_loss

        loss = l1_ssim_loss(state["image"], state["target"], case["lam"])
        return [loss, torch.autograd.grad(loss, state["image"])[0]]
    if kind == "adam":
        opt = state["opt"]
        opt.step(visibility=state["visibility"])
        ps = list(state["params"].values())
        return {"params": [t.detach() for t in ps], "m": [opt.state[t]["exp_avg"] for t in ps],
                "v": [opt.state[t]["exp_avg_sq"] for t in ps]}
    if kind == "fit":
        from gs2d import bin_gaussians, rasterize

        model, h, w = state["model"], case["height"], case["width"]
        means, conic, color, opacity, _, radii = model.activated_fused()
        bins = bin_gaussians(means, radii, model.depth, h, w)
        image = rasterize(means, conic, color, opacity, bins, backend="splat")
        loss = ((image - state["target"]) ** 2).mean()
        return [image, *torch.autograd.grad(loss, list(model.parameters()))]
    if kind == "toy2d":
        from gs2d import bin_gaussians, rasterize

        means, conic, color, opacity = state["leaves"]
        bins = bin_gaussians(means, state["radii"], state["depth"], case["height"], case["width"])
        image = rasterize(means, conic, color, opacity, bins, backend=case["backend"])
        return [image, bins.ranges, *torch.autograd.grad(image, state["leaves"], state["grad"])]
    from splat2d import render

    image = render(*state["leaves"], case["height"], case["width"], mode=case["mode"])
    return [image, *torch.autograd.grad(image, state["leaves"], state["grad"])]


# ---- what a pass cannot do without ------------------------------------------------------------


def work(case):
    """Each input read once, each output written once. The blended (pixel, Gaussian) pairs depend
    on the scene, so no operations are counted for the rasterizers."""
    kind = case["kind"]
    px = case.get("width", 0) * case.get("height", 0)
    if kind in ("view", "infer", "step"):
        par = case["n"] * (44 + 12 * (case["degree"] + 1) ** 2)  # float32 parameters
        if kind == "view":  # parameters, their gradients, tiles touched, image, alpha, image gradient
            return {"bytes": 2 * par + 4 * case["n"] * (1 + case["stats"]) + 28 * px, "flops": 0}
        if kind == "infer":
            return {"bytes": par + 16 * px, "flops": 0}
        return {"bytes": 6 * par + 24 * px, "flops": 0}  # parameters and both moments in and out, image, target
    if kind == "loss":  # both images, the gradient; five 11-tap windows in two passes, forward and backward
        c = case["channels"] * px
        return {"bytes": 12 * c, "flops": c * 2 * 8 * 22}
    if kind == "adam":
        k = (case["degree"] + 1) ** 2
        rest, one = 3 * (k - 1) * case["n"], 14 * case["n"]
        return {"bytes": case["visible"] * (28 * one + (20 if case["lowp"] else 28) * rest)
                + (4 * case["n"] if case["visible"] < 1.0 else 0), "flops": 12 * (rest + one)}
    size = 8 if case.get("f64") else 4
    per = 9 if kind != "fit" else 10  # parameters in, gradients out; image, its gradient or the target
    return {"bytes": size * (2 * per * case["n"] + 6 * px), "flops": 0}


def tolerance(case):
    """Measured against exact() and between runs (float32 atomics add in any order). A pixel's
    alpha >= 1/255 decision within rounding of the threshold moves single values far more than the
    norm: the "max" entries. The 3D gradients go through the inverse of the 2D covariance, which
    amplifies float32 rounding for elongated splats (up to 1.3e-3 from 64 bits at 3M)."""
    kind = case["kind"]
    if kind == "view":
        return {"rel": 1e-3, "max": 0.2}
    if kind == "step":  # the L1 term's sign flips where image and target agree to rounding
        return {"rel": 1e-3, "max": 0.2}
    if kind == "infer":
        return {"rel": 2e-5, "max": 0.02}
    if kind == "loss":
        return {"rel": 2e-6, "max": 1e-4}
    if kind == "adam":
        return {"rel": 1e-2, "max": 0.05} if case["lowp"] else {"rel": 3e-7, "max": 1e-5}
    if kind == "phase0" and case["f64"]:
        return {"rel": 1e-9, "max": 1e-6}
    return {"rel": 1e-4, "max": 0.02}


# ---- 64 bits ----------------------------------------------------------------------------------


def _tile_lists(x0, x1, y0, y1, order, w, h):
    """Ids of the splats whose pixel box [x0, x1] x [y0, y1] meets each tile, in the order given,
    and the lists' bounds on the host."""
    tx, ty = (w + TILE - 1) // TILE, (h + TILE - 1) // TILE
    a0, a1 = (x0 // TILE).clamp(0, tx - 1)[order], (x1 // TILE).clamp(0, tx - 1)[order]
    b0, b1 = (y0 // TILE).clamp(0, ty - 1)[order], (y1 // TILE).clamp(0, ty - 1)[order]
    nx = (a1 - a0 + 1).clamp(min=0)
    count = nx * (b1 - b0 + 1).clamp(min=0)
    item = torch.repeat_interleave(torch.arange(order.numel(), device=DEV), count)
    k = torch.arange(item.numel(), device=DEV) - (torch.cumsum(count, 0) - count)[item]
    tile = (b0[item] + k // nx[item]) * tx + a0[item] + k % nx[item]
    tile, perm = torch.sort(tile, stable=True)
    bounds = torch.searchsorted(tile, torch.arange(tx * ty + 1, device=DEV)).tolist()
    return order[item[perm]], bounds


def _blend64(mean, shape, opacity, color, ids_bounds, w, h, rules, bg=(0.0, 0.0, 0.0), grad=None):
    """Front-to-back blending tile by tile in float64. rules: "3d", "toy2d" or "phase0". grad [3, H, W]
    or a function image -> grad. Returns the image, 1 - T, and (with grad) the gradients with respect
    to mean, shape, opacity and colour and of |dL/dmean|."""
    ids_all, bounds = ids_bounds
    f = torch.float64
    off = 0.0 if rules == "toy2d" else 0.5
    bg = torch.tensor(bg, dtype=f, device=DEV)
    image, final = torch.empty(3, h, w, dtype=f, device=DEV), torch.ones(h, w, dtype=f, device=DEV)
    tx = (w + TILE - 1) // TILE
    out = [torch.zeros_like(t) for t in (mean, shape, opacity, color, mean)]
    ends = {}

    def tile(t, backward):
        x0, y0 = (t % tx) * TILE, (t // tx) * TILE
        x1, y1 = min(x0 + TILE, w), min(y0 + TILE, h)
        s, e = bounds[t], bounds[t + 1]
        if s == e:
            if not backward:
                image[:, y0:y1, x0:x1] = bg[:, None, None]
            return
        X = (torch.arange(x0, x1, dtype=f, device=DEV) + off)[None, None, :]
        Y = (torch.arange(y0, y1, dtype=f, device=DEV) + off)[None, :, None]

        def evaluate(ids):
            m, p, o = mean[ids], shape[ids], opacity[ids][:, None]
            dx, dy = (m[:, 0, None, None] - X), (m[:, 1, None, None] - Y)
            dx, dy = (v.expand(-1, y1 - y0, x1 - x0).reshape(len(ids), -1) for v in (dx, dy))
            s0, s1, s2 = p[:, 0:1], p[:, 1:2], p[:, 2:3]
            if rules == "phase0":
                a_, b_ = s0 * dx + s1 * dy, s2 * dy
                power = -0.5 * (a_ * a_ + b_ * b_)
            else:
                a_ = b_ = None
                power = -0.5 * (s0 * dx * dx + s2 * dy * dy) - s1 * dx * dy
            raw = o * torch.exp(power.clamp(max=0.0))
            alpha = raw if rules == "3d" else raw.clamp(max=0.99)
            ok = alpha >= 1.0 / 255.0
            if rules == "toy2d":
                ok = ok & (power <= 0)
            return torch.where(ok, alpha, 0.0), ok, raw, o, dx, dy, s0, s1, s2, a_, b_

        if not backward:  # the part of the list after which every pixel of the tile has stopped
            T = torch.ones((), dtype=f, device=DEV)
            ends[t] = e
            for c0 in range(s, e - 1024, 1024):
                T = T * torch.prod(1.0 - evaluate(ids_all[c0:c0 + 1024])[0], 0)
                if float(T.max()) < 1e-4:
                    ends[t] = c0 + 1024
                    break
        ids = ids_all[s:ends[t]]
        c = color[ids]
        alpha, ok, raw, o, dx, dy, s0, s1, s2, a_, b_ = evaluate(ids)
        after = torch.cumprod(1.0 - alpha, 0)
        before = torch.cat([torch.ones_like(after[:1]), after[:-1]], 0)
        live = ok & ((after if rules == "toy2d" else before) >= 1e-4)
        alpha = torch.where(live, alpha, 0.0)
        weight = alpha * before
        T = torch.prod(1.0 - alpha, 0)
        if not backward:
            image[:, y0:y1, x0:x1] = (c.T @ weight + bg[:, None] * T).reshape(3, y1 - y0, x1 - x0)
            final[y0:y1, x0:x1] = T.reshape(y1 - y0, x1 - x0)
            return
        gp = grad[:, y0:y1, x0:x1].reshape(3, -1)
        gc = c @ gp
        v = weight * gc
        behind = v.sum(0) - torch.cumsum(v, 0) + T * (bg @ gp)
        da = before * gc - behind / (1.0 - alpha).clamp(min=1e-6)
        dpow = torch.where(live if rules == "3d" else live & (raw <= 0.99), alpha * da, 0.0)
        if rules == "phase0":  # a = l0 dx + l1 dy, b = l2 dy; here dx, dy are mean - pixel
            gx, gy = -dpow * a_ * s0, -dpow * (a_ * s1 + b_ * s2)
            gs = (-dpow * a_ * dx, -dpow * a_ * dy, -dpow * b_ * dy)
        else:
            gx, gy = -dpow * (s0 * dx + s1 * dy), -dpow * (s1 * dx + s2 * dy)
            gs = (-0.5 * dpow * dx * dx, -dpow * dx * dy, -0.5 * dpow * dy * dy)
        out[0].index_add_(0, ids, torch.stack([gx.sum(1), gy.sum(1)], -1))
        out[1].index_add_(0, ids, torch.stack([t.sum(1) for t in gs], -1))
        out[2].index_add_(0, ids, dpow.sum(1) / o[:, 0])
        out[3].index_add_(0, ids, weight @ gp.T)
        out[4].index_add_(0, ids, torch.stack([gx.abs().sum(1), gy.abs().sum(1)], -1))

    tiles = range(len(bounds) - 1)
    for t in tiles:
        tile(t, False)
    if grad is None:
        return image, 1.0 - final, None
    if callable(grad):
        grad = grad(image)
    for t in tiles:
        tile(t, True)
    return image, 1.0 - final, out


_SH = (0.28209479177387814, 0.4886025119029199, 1.0925484305920792, 0.31539156525252005, 0.5462742152960396,
       0.5900435899266435, 2.890611442640554, 0.4570457994644658, 0.3731763325901154, 1.445305721320277)


def _basis64(d, K):
    x, y, z = d.unbind(1)
    b = [torch.full_like(x, _SH[0])]
    if K >= 4:
        b += [-_SH[1] * y, _SH[1] * z, -_SH[1] * x]
    if K >= 9:
        b += [_SH[2] * x * y, -_SH[2] * y * z, _SH[3] * (3 * z * z - 1), -_SH[2] * x * z, _SH[4] * (x * x - y * y)]
    if K >= 16:
        b += [-_SH[5] * y * (3 * x * x - y * y), _SH[6] * x * y * z, -_SH[7] * y * (5 * z * z - 1),
              _SH[8] * z * (5 * z * z - 3), -_SH[7] * x * (5 * z * z - 1), _SH[9] * z * (x * x - y * y),
              -_SH[5] * x * (x * x - 3 * y * y)]
    return torch.stack(b, 1)


def _project64(m, ls, q, logit, sh, cam, antialias):
    """Screen-space means, conics, opacities, colours, 2D covariances and depths, differentiable."""
    vm = cam["viewmat"].double()
    R, t = vm[:3, :3].to(DEV), vm[:3, 3].to(DEV)
    fx, fy, cx, cy = (float(cam["K"][i, j]) for i, j in ((0, 0), (1, 1), (0, 2), (1, 2)))
    v = m @ R.T + t
    z = v[:, 2]
    x, y = v[:, 0] / z, v[:, 1] / z
    xc = x.clamp(-1.3 * cx / fx, 1.3 * (cam["W"] - cx) / fx)  # the Jacobian's clamp to 1.3 of the frustum
    yc = y.clamp(-1.3 * cy / fy, 1.3 * (cam["H"] - cy) / fy)
    q = q / q.norm(dim=1, keepdim=True)
    r, i, j, k = q.unbind(1)
    rot = torch.stack([1 - 2 * (j * j + k * k), 2 * (i * j - r * k), 2 * (i * k + r * j), 2 * (i * j + r * k),
                       1 - 2 * (i * i + k * k), 2 * (j * k - r * i), 2 * (i * k - r * j), 2 * (j * k + r * i),
                       1 - 2 * (i * i + j * j)], 1).reshape(-1, 3, 3)
    M = rot * torch.exp(ls)[:, None, :]
    o0 = torch.zeros_like(z)
    J = torch.stack([fx / z, o0, -fx * xc / z, o0, fy / z, -fy * yc / z], 1).reshape(-1, 2, 3)
    A = (J @ R) @ M
    xx, xy, yy = (A[:, 0] ** 2).sum(1), (A[:, 0] * A[:, 1]).sum(1), (A[:, 1] ** 2).sum(1)
    a, c = xx + 0.3, yy + 0.3
    det = a * c - xy * xy
    o = torch.sigmoid(logit)
    if antialias:
        o = o * torch.sqrt(((xx * yy - xy * xy) / det).clamp(min=0.0))
    d = m + (R.T @ t)
    d = d / d.norm(dim=1, keepdim=True)
    color = ((_basis64(d, sh.shape[1])[:, :, None] * sh).sum(1) + 0.5).clamp(min=0.0)
    return (torch.stack([fx * x + cx, fy * y + cy], 1), torch.stack([c / det, -xy / det, a / det], 1), o, color,
            torch.stack([a, c], 1), z, torch.sigmoid(logit))


def _touches64(mean, conic, o, reach, w, h):
    """Whether the alpha >= 1/255 ellipse crosses a column of pixel centres of the image between the
    first and last rows of pixel centres of some row of tiles (the rule of the tile lists)."""
    A, B, C = conic.unbind(1)
    t2 = 2.0 * torch.log((255.0 * o).clamp(min=1.0))
    det = A * C - B * B
    xlo, xhi = torch.ceil(mean[:, 0] - reach[:, 0] - 0.5).clamp(min=0), torch.floor(mean[:, 0] + reach[:, 0] - 0.5)
    ylo, yhi = torch.ceil(mean[:, 1] - reach[:, 1] - 0.5).clamp(min=0), torch.floor(mean[:, 1] + reach[:, 1] - 0.5)
    xhi, yhi = xhi.clamp(max=w - 1), yhi.clamp(max=h - 1)
    top = torch.sqrt(t2 * A / det)
    right = -(B / C) * torch.sqrt(t2 * C / det)  # the row of the ellipse's rightmost point
    hit = torch.zeros_like(o, dtype=torch.bool)
    for y in range(0, h, TILE):
        v0 = torch.maximum(ylo.clamp(min=y) + 0.5 - mean[:, 1], -top)
        v1 = torch.minimum(yhi.clamp(max=y + TILE - 1) + 0.5 - mean[:, 1], top)
        r, l = (torch.minimum(torch.maximum(s * right, v0), v1) for s in (1.0, -1.0))
        xr = mean[:, 0] + (torch.sqrt((t2 * A - det * r * r).clamp(min=0)) - B * r) / A
        xl = mean[:, 0] - (torch.sqrt((t2 * A - det * l * l).clamp(min=0)) + B * l) / A
        first, last = torch.maximum(torch.ceil(xl - 0.5), xlo), torch.minimum(torch.floor(xr - 0.5), xhi)
        hit |= (v0 <= v1) & (first <= last)
    return hit


def _view64(model, cam, bg, antialias, grad):
    """image, alpha, gradients with respect to the model (or None) and the mean gradients' parts."""
    leaves = [t.detach().double().requires_grad_(grad is not None) for t in model]
    with torch.set_grad_enabled(grad is not None):
        mean, conic, o, color, cov, z, o_raw = _project64(*leaves, cam, antialias)
    scr = [t.detach() for t in (mean, conic, o, color)]
    w, h = cam["W"], cam["H"]
    reach = torch.sqrt(2.0 * torch.log((255.0 * scr[2]).clamp(min=1.0))[:, None] * cov.detach())
    lo, hi = torch.floor(scr[0] - reach - 0.5).long(), torch.ceil(scr[0] + reach - 0.5).long()
    seen = (z > cam["near"]) & (z < cam["far"]) & (o_raw >= 1.0 / 255.0) & (scr[2] >= 1.0 / 255.0)
    seen &= (hi[:, 0] >= 0) & (hi[:, 1] >= 0) & (lo[:, 0] < w) & (lo[:, 1] < h)
    order = torch.nonzero(seen)[:, 0]
    order = order[torch.sort(z.detach()[order], stable=True)[1]]
    lists = _tile_lists(lo[:, 0], hi[:, 0], lo[:, 1], hi[:, 1], order, w, h)
    image, alpha, out = _blend64(*scr, lists, w, h, "3d", bg, grad)
    if grad is None:
        return image, alpha, None, None
    seen = seen & _touches64(scr[0], scr[1], scr[2], reach, w, h)
    grads = torch.autograd.grad([mean, conic, o, color], leaves, out[:4])
    return image, alpha, grads, (out[0], out[4], seen)


def _ssim64(x, y):
    k = torch.arange(11, dtype=torch.float64, device=DEV) - 5
    k = torch.exp(-k * k / (2 * 1.5 ** 2))
    k = k / k.sum()

    def blur(t):
        t = torch.nn.functional.conv2d(t[:, None], k.reshape(1, 1, 1, 11), padding=(0, 5))
        return torch.nn.functional.conv2d(t, k.reshape(1, 1, 11, 1), padding=(5, 0))[:, 0]

    mx, my = blur(x), blur(y)
    vx, vy, vxy = blur(x * x) - mx * mx, blur(y * y) - my * my, blur(x * y) - mx * my
    c1, c2 = 0.01 ** 2, 0.03 ** 2
    return (((2 * mx * my + c1) * (2 * vxy + c2)) / ((mx * mx + my * my + c1) * (vx + vy + c2))).mean()


def _loss64(image, target, lam):
    """The loss and its image gradient."""
    x = image.detach().double().requires_grad_(True)
    y = target.double()
    with torch.enable_grad():
        loss = (1.0 - lam) * (x - y).abs().mean() + lam * (1.0 - _ssim64(x, y))
        return loss.detach(), torch.autograd.grad(loss, x)[0]


def _adam64(opt, names, params, grads, seen):
    """Updated parameters and moments, a row at a time where `seen` masks rows."""
    got = ([], [], [])
    for k, p, g in zip(names, params, grads):
        s = opt.state[p]
        m0, v0, p0, g = s["exp_avg"].double(), s["exp_avg_sq"].double(), p.detach().double(), g.double()
        t = s["step"] + 1
        m, v = 0.9 * m0 + 0.1 * g, 0.999 * v0 + 0.001 * g * g
        new = p0 - LEARNING_RATES[k] / (1 - 0.9 ** t) * m / (torch.sqrt(v) / math.sqrt(1 - 0.999 ** t) + 1e-15)
        if seen is not None:
            on = seen.reshape(-1, *[1] * (p.dim() - 1))
            new, m, v = (torch.where(on, a, b) for a, b in ((new, p0), (m, m0), (v, v0)))
        for to, x in zip(got, (new, m, v)):
            to.append(x)
    return got


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    w, h = case.get("width"), case.get("height")
    if kind in ("view", "infer", "step"):
        _, model, cam = _view_inputs(case, seed)
        if kind == "infer":
            return list(_view64(model, cam, (0.1, 0.2, 0.3), case["antialias"], None)[:2])
        if kind == "view":
            image, alpha, grads, (g2, ga, _) = _view64(model, cam, (0.1, 0.2, 0.3), case["antialias"],
                                                          s["grad"].double())
            gm, gls, gq, go, gsh = grads
            stats = None
            if case["stats"]:
                half = torch.tensor([0.5 * w, 0.5 * h], dtype=torch.float64, device=DEV)
                # (the count's row follows the float32 tile rule, as the tile counts do)
                stats = [None, (g2 * half).norm(dim=1), (ga * half).norm(dim=1)][:case["stats"]]
            return {"image": image, "alpha": alpha, "touched": None,
                    "grads": [gm, gls, gq, go, *((gsh[:, :1], gsh[:, 1:]) if case["split"] else (gsh,))],
                    "stats": stats}
        got = {}

        def loss_grad(image):
            got["loss"], g = _loss64(image, s["target"], 0.2)
            return g

        image, _, (gm, gls, gq, go, gsh), (_, _, seen) = _view64(model, cam, (0.0, 0.0, 0.0), False, loss_grad)
        new, m, _ = _adam64(s["opt"], list(s["params"]), list(s["params"].values()),
                            [gm, gls, gq, gsh[:, :1], gsh[:, 1:], go], seen if case["masked"] else None)
        return {"image": image, "loss": got["loss"], "params": new, "m": m}
    if kind == "loss":
        return list(_loss64(s["image"], s["target"], case["lam"]))
    if kind == "adam":
        vis = None if s["visibility"] is None else s["visibility"] > 0
        names, ps = list(s["params"]), list(s["params"].values())
        new, m, v = _adam64(s["opt"], names, ps, [p.grad for p in ps], vis)
        if case["lowp"]:  # stochastically rounded moments have no value of their own
            for x in (m, v):
                x[names.index("sh_rest")] = None
        return {"params": new, "m": m, "v": v}
    if kind in ("fit", "toy2d"):
        from gs2d.params import radii_from_cov

        _, xy, log_scale, theta, rgb, logit, depth = _gaussians2d(case, seed)
        raw = [t.double().requires_grad_(True) for t in (xy, log_scale, theta, rgb, logit)]
        with torch.enable_grad():
            c, sn = torch.cos(raw[2]), torch.sin(raw[2])
            v = torch.exp(2 * raw[1])
            xx, yy = c * c * v[:, 0] + sn * sn * v[:, 1], sn * sn * v[:, 0] + c * c * v[:, 1]
            xy_ = c * sn * (v[:, 0] - v[:, 1])
            det = xx * yy - xy_ * xy_
            act = [raw[0], torch.stack([yy, -xy_, xx], 1) / det[:, None], torch.sigmoid(raw[4]), torch.sigmoid(raw[3])]
        if kind == "toy2d":  # the activated float32 values are the inputs
            m_, cn, col, op = (t.detach().double() for t in s["leaves"])
            scr, radii, grad = [m_, cn, op, col], s["radii"], s["grad"].double()
        else:
            scr, grad = [t.detach() for t in act], None
            radii = radii_from_cov(torch.stack([xx, xy_, yy], 1).detach().float())
        r = radii.double()
        mx, my = xy.double().unbind(1)
        # tiles [trunc((m - r) / 16), trunc((m + r + 15) / 16)) of the 3-sigma square
        tw, th = (w + TILE - 1) // TILE, (h + TILE - 1) // TILE
        b = [torch.trunc(t / TILE).long() for t in (mx - r, mx + r + 15, my - r, my + r + 15)]
        box = (b[0].clamp(0, tw), b[1].clamp(0, tw), b[2].clamp(0, th), b[3].clamp(0, th))
        has = torch.nonzero((r > 0) & (box[1] > box[0]) & (box[3] > box[2]))[:, 0]
        order = has[torch.sort(depth[has], stable=True)[1]]
        lists = _tile_lists(box[0] * TILE, box[1] * TILE - 1, box[2] * TILE, box[3] * TILE - 1, order, w, h)
        if kind == "fit":
            y = s["target"].double()
            image, _, out = _blend64(*scr, lists, w, h, "toy2d", grad=lambda im: 2.0 * (im - y) / im.numel())
            return [image, *torch.autograd.grad(act, raw, out[:4])]
        image, _, out = _blend64(*scr, lists, w, h, "toy2d", grad=grad)
        return [image, None, out[0], out[1], out[3], out[2]]
    *params, g = _phase0_inputs(case, seed)
    means, chol, logit, colors = (t.double() for t in params)
    o = torch.sigmoid(logit)
    reach = torch.sqrt(2.0 * torch.log((255.0 * o).clamp(min=1.0)))
    ex = reach * torch.sqrt(1.0 / chol[:, 0] ** 2 + (chol[:, 1] / (chol[:, 0] * chol[:, 2])) ** 2)
    ey = reach / chol[:, 2].abs()
    x0, x1 = torch.floor(means[:, 0] - ex - 0.5).long(), torch.ceil(means[:, 0] + ex - 0.5).long()
    y0, y1 = torch.floor(means[:, 1] - ey - 0.5).long(), torch.ceil(means[:, 1] + ey - 0.5).long()
    order = torch.nonzero((reach > 0) & (x1 >= 0) & (x0 < w) & (y1 >= 0) & (y0 < h))[:, 0]
    lists = _tile_lists(x0, x1, y0, y1, order, w, h)
    image, _, out = _blend64(means, chol, o, colors, lists, w, h, "phase0", grad=g.double().permute(2, 0, 1))
    return [image.permute(1, 2, 0), out[0], out[1], out[2] * o * (1.0 - o), out[3]]
