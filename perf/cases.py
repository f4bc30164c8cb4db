"""The work this framework is timed on: frames, gradients, training steps, density control and
the key sort, through the package's public entry points (render_, backward_, Trainer, ...).

listed() names the cases, draw() makes more of the same ranges, prepare() makes a case's inputs
on the GPU from a seed, run() is one pass, work() the bytes and operations a pass needs at least,
tolerance() what another correct float32 implementation may differ by, and exact() the same
results in 64 bits from plain torch.
"""
import math

import numpy as np
import torch

from __graft_entry__ import load_package

load_package()
from tdgs_amd import abi, core, host, training  # noqa: E402

DEV = "cuda:0"

# Scenes: "ball" is one object, means N(0, 1) seen from distance 4 at 60 degrees; "room" is a
# 20 m box with a dense core, seen from distance 6 at 50 degrees. Log-scales are normal.
SCENES = {
    "ball": {"radius": 4.0, "fov": 60.0, "mu": -3.5, "sigma": 0.4},
    "room": {"radius": 6.0, "fov": 50.0, "mu": -4.0, "sigma": 0.6},
    "dense": {"radius": 6.0, "fov": 50.0, "mu": -2.5, "sigma": 0.8},
}


def listed():
    return [
        # a thumbnail of a small object: everything is launch and host latency; counts read back
        {"name": "render_10k_256", "what": "render", "scene": "ball", "n": 10_000, "w": 256, "h": 256, "degree": 0,
         "tw": 16, "th": 16, "host_counts": True},
        # one frame of an orbit video, a million Gaussians at full HD, nothing read back
        {"name": "render_1m_1080p", "what": "render", "scene": "room", "n": 1_000_000, "w": 1920, "h": 1080,
         "degree": 3, "tw": 16, "th": 16, "host_counts": False},
        # a viewer's frame of a loaded model: covariances and opacities given, antialiasing on,
        # depth too, and the 8-bit image it shows
        {"name": "view_300k_720p", "what": "view", "scene": "room", "n": 300_007, "w": 1280, "h": 720, "degree": 3,
         "tw": 16, "th": 16},
        # render! and backward! for a loss of the caller's own, the defaults
        {"name": "grad_200k_800", "what": "grad", "scene": "ball", "n": 200_000, "w": 800, "h": 800, "degree": 3,
         "tw": 16, "th": 16, "aa": False, "filter": False, "layout": "interleaved"},
        # the same in the middle of the spherical harmonics' ramp, on a ragged image, with
        # antialiasing, the boundary filter, tall tiles and the four gradient arrays
        {"name": "grad_60k_ragged", "what": "grad", "scene": "room", "n": 60_013, "w": 979, "h": 546, "degree": 1,
         "tw": 16, "th": 32, "aa": True, "filter": True, "layout": "reference"},
        # training a small model at thumbnail size, as at the start of a run (constant colours)
        {"name": "step_20k_400", "what": "step", "scene": "ball", "n": 20_000, "w": 400, "h": 400, "degree": 0,
         "tw": 16, "th": 16},
        # training at the size of a usual photo set, before density control has grown the model
        {"name": "step_500k_1297x840", "what": "step", "scene": "room", "n": 500_000, "w": 1297, "h": 840,
         "degree": 3, "tw": 16, "th": 16},
        # training a grown model at full HD
        {"name": "step_1m_1080p", "what": "step", "scene": "room", "n": 1_000_000, "w": 1920, "h": 1080, "degree": 3,
         "tw": 16, "th": 16},
        # the training loss and its gradient by itself (evaluation of the losses)
        {"name": "loss_1080p", "what": "loss", "w": 1920, "h": 1080, "weight": 0.2},
        # one densification: clone, split and prune parameters and moments
        {"name": "density_500k", "what": "density", "n": 500_000, "degree": 3, "share": 0.08},
        # the key sort by itself, the keys of one full HD frame
        {"name": "sort_6m", "what": "sort", "n": 6_150_000, "tiles": 8160},
        # the largest: three million large Gaussians at 4K, hundreds of millions of keys, both ways
        {"name": "grad_3m_4k", "what": "grad", "scene": "dense", "n": 3_000_000, "w": 3840, "h": 2160, "degree": 3,
         "tw": 16, "th": 32, "aa": False, "filter": False, "layout": "interleaved"},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng):
    """An image from a thumbnail to full HD, any aspect ratio between 1:1 and 2:1, odd sides too."""
    w = _log_uniform(rng, 200, 1920)
    return w, max(120, min(1080, int(w / rng.uniform(1.0, 2.0))))


def draw(rng):
    what = rng.choice(["render", "render", "view", "grad", "grad", "step", "step", "loss", "density", "sort"])
    w, h = _size(rng)
    n = _log_uniform(rng, 3_000, 1_200_000)
    case = {"what": what, "scene": rng.choice(["ball", "room"]), "n": n, "w": w, "h": h,
            "degree": rng.choice([0, 1, 2, 3, 3, 3]), "tw": 16, "th": rng.choice([16, 16, 32])}
    if what == "render":
        case["host_counts"] = rng.choice([True, False])
    elif what == "grad":
        case.update(aa=rng.choice([False, True]), filter=rng.choice([False, False, True]),
                    layout=rng.choice(["interleaved", "reference"]))
        if rng.random() < 0.25:
            case.update(tw=8, th=8)
    elif what == "loss":
        case = {"what": "loss", "w": w, "h": h, "weight": rng.choice([0.2, 0.2, 1.0])}
    elif what == "density":
        case = {"what": "density", "n": n, "degree": case["degree"], "share": round(rng.uniform(0.0, 0.3), 3)}
    elif what == "sort":
        case = {"what": "sort", "n": _log_uniform(rng, 3_000, 20_000_000), "tiles": _log_uniform(rng, 16, 30_000)}
    return case


# ------------------------------------------------------------------------------------
# Inputs
# ------------------------------------------------------------------------------------

def _scene(case, seed):
    """Parameters on the GPU: means and opacity logits (n, 4), log-scales, quaternions, SH (n, 3, h)."""
    g = torch.Generator(device=DEV)
    g.manual_seed(1_000_003 * (int(seed) + 1))
    s, n, hh = SCENES[case["scene"]], case["n"], (case["degree"] + 1) ** 2

    def randn(*shape):
        return torch.randn(shape, generator=g, device=DEV)

    if case["scene"] == "ball":
        means = randn(n, 3)
    else:   # half the Gaussians over the room, half in its core, in any order
        far = torch.rand((n, 3), generator=g, device=DEV) * 20 - 10
        pick = torch.rand((n, 1), generator=g, device=DEV) < 0.5
        means = torch.where(pick, far, 1.5 * randn(n, 3))
    mo = torch.cat([means, 1.5 * randn(n, 1)], dim=1)
    scaling = s["mu"] + s["sigma"] * randn(n, 3)
    q = randn(n, 4)
    q = q / q.norm(dim=1, keepdim=True)
    sh = 0.05 * randn(n, 3, hh)
    sh[:, :, 0] = 0.3 * randn(n, 3)
    return mo, scaling, q, sh


def _camera(case, seed, k=0):
    """Camera k of the case's orbit (the seed sets where the orbit starts)."""
    s = SCENES[case["scene"]]
    az = 2 * math.pi * (((seed * 0.6180339887) % 1.0) + k / 8)
    el = math.radians(-15 + 30 * ((seed * 0.7548776662 + k * 0.5698402910) % 1.0))
    pos = s["radius"] * np.array([math.cos(el) * math.sin(az), -math.sin(el), -math.cos(el) * math.cos(az)])
    return host.look_at_camera(case["w"], case["h"], s["fov"], pos)


def _options(case, cam):
    view = case["what"] == "view"
    return host.RenderOptions.for_camera(
        cam, case["degree"], use_antialiasing=view or case.get("aa", False),
        clip_mode=abi.TDGS_CLIP_FILTER if case.get("filter") else abi.TDGS_CLIP_CLAMP,
        background_color=(0.9, 0.9, 0.9) if view else (0.0, 0.0, 0.0))


def _image(case, seed):
    """A target image (w, h, 3): smooth shapes and noise, values in [0, 1]."""
    g = torch.Generator(device=DEV)
    g.manual_seed(7_000_003 * (int(seed) + 1))
    w, h = case["w"], case["h"]
    x = torch.linspace(0, 1, w, device=DEV)[:, None, None]
    y = torch.linspace(0, 1, h, device=DEV)[None, :, None]
    f = 2 + 6 * torch.rand((2, 1, 1, 3), generator=g, device=DEV)
    smooth = 0.5 + 0.3 * torch.sin(6.2832 * (f[0] * x + f[1] * y))
    return (smooth + 0.1 * torch.randn((w, h, 3), generator=g, device=DEV)).clamp(0, 1).contiguous()


def _image_grad(case, seed):
    """The gradient of a mean over the pixels, as a loss of the caller's own gives it."""
    g = torch.Generator(device=DEV)
    g.manual_seed(9_000_011 * (int(seed) + 1))
    shape = (case["w"], case["h"], 3)
    return torch.randn(shape, generator=g, device=DEV) / (case["w"] * case["h"] * 3)


def _moments(case, seed, n, hh):
    """Adam moments of a run some hundred steps old: second moments of gradients of a mean over
    the pixels, first moments a few times smaller than their roots."""
    g = torch.Generator(device=DEV)
    g.manual_seed(11_000_027 * (int(seed) + 1))

    def pair(scale, *shape):
        r = scale * (0.2 + torch.rand(shape, generator=g, device=DEV))
        return torch.stack([0.3 * r * torch.randn(shape, generator=g, device=DEV), r * r], dim=-1).contiguous()

    return {"means": pair(2e-7, n, 3), "opacity": pair(5e-8, n), "scaling": pair(1e-7, n, 3),
            "rotation": pair(3e-8, n, 4), "sh": pair(2e-8, n, 3, hh)}


UPDATES = 400   # optimizer steps before the timed ones
WEIGHT = 0.2    # of D-SSIM in the training loss


def _training_options(case, lr_steps=30_000):
    """3DGS defaults without density control, opacity resets or SH growth in the timed steps."""
    return training.TrainingOptions.for_scene(
        1.1 * SCENES[case.get("scene", "room")]["radius"], loss_dssim_vs_L1_weight=WEIGHT,
        nb_lr_annealing_steps=lr_steps, adc_start_iteration_nb=10 ** 9, adc_final_iteration_nb=10 ** 9,
        opacity_reset_interval=10 ** 9, sh_degree_increase_interval=10 ** 9)


def _set_moments(optimizer, m):
    o = optimizer.moments
    o.means, o.opacity, o.scaling, o.rotation, o.sh = m["means"], m["opacity"], m["scaling"], m["rotation"], m["sh"]


def prepare(case, seed):
    what = case["what"]
    if what == "loss":
        rgb, gt = _image(case, seed), _image(case, seed + 1)
        rgb = (0.7 * gt + 0.3 * rgb).contiguous()
        temp = torch.empty(int(core.lib().tdgs_loss_temp_bytes(case["w"], case["h"])), dtype=torch.uint8, device=DEV)
        return {"case": case, "rgb": rgb, "gt": gt, "grad": torch.empty_like(rgb),
                "sums": torch.zeros(2, dtype=torch.float64, device=DEV), "temp": temp}
    if what == "sort":
        g = torch.Generator(device=DEV)
        g.manual_seed(13_000_027 * (int(seed) + 1))
        n, tiles = case["n"], case["tiles"]
        tile = torch.randint(1, tiles + 1, (n,), generator=g, device=DEV)
        depth = (2 + 10 * torch.rand(n, generator=g, device=DEV)).view(torch.int32).to(torch.int64)
        return {"case": case, "keys": (tile << 32) | depth, "end_bit": 33 + int(math.floor(math.log2(tiles))),
                "values": torch.arange(1, n + 1, dtype=torch.int32, device=DEV)}
    if what == "density":
        c = {**case, "scene": "room"}
        mo, scaling, q, sh = _scene(c, seed)
        options = _training_options(c)
        n = case["n"]
        g = torch.Generator(device=DEV)
        g.manual_seed(17_000_023 * (int(seed) + 1))
        order = torch.randperm(n, generator=g, device=DEV)
        pruned, over = order[:n // 200], order[n // 200:n // 200 + int(case["share"] * n)]
        mo[:, 3].clamp_(min=-5.0)   # (pruned below -5.3)
        mo[pruned, 3] = -6.0
        gaussians = core.TrainableGaussiansVector(mo, scaling, q, sh)
        optimizer = training.AdamOptimizer(gaussians, options, update_count=UPDATES)
        _set_moments(optimizer, _moments(c, seed, case["n"], sh.shape[2]))
        adc = training.AdaptiveDensityControlBuffers(case["n"], 0)
        counts = torch.randint(1, 100, (n,), generator=g, device=DEV, dtype=torch.int32)
        mean = options.densification_mean2d_grad_norm_threshold_ndc * (0.1 + 0.8 * torch.rand(n, generator=g, device=DEV))
        mean[over] *= 20
        adc.accum.copy_(mean * counts)
        adc.counts.copy_(counts)
        return {"case": case, "gaussians": gaussians, "optimizer": optimizer, "moments": optimizer.moments,
                "adc": adc, "options": options, "seed": int(seed)}
    cam = _camera(case, seed)
    tiling = host.Tiling.for_camera(cam, case["tw"], case["th"])
    options = _options(case, cam)
    mo, scaling, q, sh = _scene(case, seed)
    if what == "step":
        gaussians = core.TrainableGaussiansVector(mo, scaling, q, sh)
        opt = _training_options(case)
        optimizer = training.AdamOptimizer(gaussians, opt, update_count=UPDATES)
        _set_moments(optimizer, _moments(case, seed, case["n"], sh.shape[2]))
        cams = [_camera(case, seed, k) for k in range(4)]
        images = [_image(case, 4 * seed + k) for k in range(4)]
        trainer = training.Trainer(gaussians, cams, images, options, tiling, opt, optimizer=optimizer,
                                   seed=int(seed) & 0xffff)
        # the key arrays of a run under way hold its largest frame
        for k in range(4):
            core.render_(trainer.render_outputs, gaussians, cams[k], tiling, options, trainer.render_buffers,
                         ctx=trainer.ctx)
        return {"case": case, "trainer": trainer}
    if what == "view":
        op = torch.sigmoid(mo[:, 3:4])
        R = _rotation(q.double())
        M = R * scaling.double().exp()[:, None, :]
        V = M @ M.transpose(1, 2)
        lower = torch.stack([V[:, 0, 0], V[:, 1, 0], V[:, 2, 0], V[:, 1, 1], V[:, 2, 1], V[:, 2, 2]], dim=1)
        gaussians = core.RenderOnlyGaussiansVector(torch.cat([mo[:, :3], op], dim=1), lower.float(), sh)
    else:
        gaussians = core.TrainableGaussiansVector(mo, scaling, q, sh)
    buffers = core.RenderBuffers(case["n"], tiling, 0)
    outputs = core.RenderOutputs.for_camera(cam, 0, include_depth=what == "view",
                                            include_last_contributing_indices=what == "grad")
    state = {"case": case, "gaussians": gaussians, "camera": cam, "tiling": tiling, "options": options,
             "buffers": buffers, "outputs": outputs}
    if what == "view":
        state["image"] = torch.empty((case["h"], case["w"], 3), dtype=torch.uint8, device=DEV)
    if what == "grad":
        state["rgb_grad"] = _image_grad(case, seed)
        state["gradients"] = core.FilteredGaussiansGradientsVector(case["n"], case["degree"], 0,
                                                                   layout=case["layout"])
    # the first frame sizes the key arrays
    core.render_(outputs, gaussians, cam, tiling, options, buffers)
    return state


# ------------------------------------------------------------------------------------
# One pass
# ------------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    what = case["what"]
    if what == "loss":
        state["sums"].zero_()
        training.loss_grad_(state["rgb"], state["gt"], state["grad"], case["weight"], state["sums"], state["temp"])
        return {"grad": state["grad"], "sums": state["sums"]}
    if what == "sort":
        keys, values = core.sort_pairs(state["keys"], state["values"], state["end_bit"])
        return {"keys": keys, "values": values}
    if what == "density":
        g, optimizer, adc, o = state["gaussians"], state["optimizer"], state["adc"], state["options"]
        optimizer.gaussians, optimizer.moments = g, state["moments"]
        n_new = training.adc_plan_(adc, g, *training.adc_plan_thresholds(1000, o))
        new = training.adaptive_density_control_(adc, g, optimizer, n_new, math.log(o.splitting_scale_factor),
                                                 state["seed"])
        m = optimizer.moments
        return {"means_opacity": new.means_opacity, "scaling": new.scaling, "rotation": new.rotation, "sh": new.sh,
                "m_means": m.means, "m_opacity": m.opacity, "m_scaling": m.scaling, "m_rotation": m.rotation,
                "m_sh": m.sh, "n": n_new}
    if what == "step":
        t = state["trainer"]
        t.training_step_()
        g, m = t.gaussians, t.optimizer.moments
        return {"rgb": t.render_outputs.rgb, "loss_sums": t.loss_sums, "rgb_grad": t.rgb_image_grad,
                "means_opacity": g.means_opacity, "scaling": g.scaling, "rotation": g.rotation, "sh": g.sh,
                "m_means": m.means, "m_opacity": m.opacity, "m_scaling": m.scaling, "m_rotation": m.rotation,
                "m_sh": m.sh}
    out, buf = state["outputs"], state["buffers"]
    core.render_(out, state["gaussians"], state["camera"], state["tiling"], state["options"], buf,
                 device_counts=what == "render" and not case["host_counts"])
    if what == "render":
        return {"rgb": out.rgb, "T": out.T}
    if what == "view":
        core.image_to_rgb8(out.rgb, out=state["image"])
        return {"rgb": out.rgb, "T": out.T, "depth": out.depth, "image": state["image"]}
    gr = state["gradients"]
    core.backward_(gr, state["rgb_grad"], out, state["gaussians"], state["camera"], state["tiling"],
                   state["options"], buf)
    # (the rows past the kept Gaussians, buf.nb_fgaussians of them, stay zero)
    return {"rgb": out.rgb, "T": out.T, "last": out.last, "kept": buf.nb_fgaussians, "mean2d": gr.mean2d,
            "opacity2d": gr.opacity, "conic": gr.licov2d, "color": gr.color, "mean": gr.mean3d,
            "opacity": gr.opacity_feature, "scaling": gr.scaling_features, "rotation": gr.rotation_features,
            "sh": gr.sh}


# ------------------------------------------------------------------------------------
# What a pass cannot do without
# ------------------------------------------------------------------------------------

def _pairs(case):
    """(share of Gaussians in view, (pixel, Gaussian) pairs with alpha >= 1 / 255 that a pixel
    meets before it is opaque), estimated from 4096 Gaussians of the case's distribution."""
    rng = np.random.Generator(np.random.PCG64(5))
    s, k = SCENES[case["scene"]], 4096
    if case["scene"] == "ball":
        m = rng.normal(size=(k, 3))
    else:
        m = np.where(rng.random((k, 1)) < 0.5, rng.uniform(-10, 10, (k, 3)), 1.5 * rng.normal(size=(k, 3)))
    a = 1 / (1 + np.exp(-1.5 * rng.normal(size=k)))
    z = m[:, 2] + s["radius"]
    f = case["w"] / 2 / math.tan(math.radians(s["fov"]) / 2)
    sig = f * np.exp(s["mu"] + s["sigma"] * rng.normal(size=(k, 2))) / np.maximum(z, 0.2)[:, None]
    sig = np.sqrt(sig * sig + 0.3)
    u, v = np.abs(f * m[:, 0] / z), np.abs(f * m[:, 1] / z)
    seen = (z > 0.2) & (a > 1 / 255) & (u < case["w"] / 2) & (v < case["h"] / 2)
    px = case["w"] * case["h"]
    area = np.where(seen, np.minimum(2 * math.pi * np.log(np.maximum(255 * a, 1)) * sig.prod(1), px), 0)
    depth = np.where(seen, np.minimum(2 * math.pi * a * (1 + a / 4) * sig.prod(1), px), 0)   # -log(1 - alpha), summed
    scale = case["n"] / k
    opaque = depth.sum() * scale / px / 9.2   # T falls below 1e-4 after 9.2
    return float(seen.mean()), float(area.sum() * scale / max(1.0, opaque))


def work(case):
    what = case["what"]
    if what == "loss":
        px = case["w"] * case["h"]
        # two images in, one out; five 22-tap filters and three back, and the SSIM map, per channel
        return {"bytes": 4 * 3 * 3 * px, "flops": 3 * px * (8 * 44 + 60)}
    if what == "sort":
        return {"bytes": 2 * 12 * case["n"], "flops": 0}
    hh = (case["degree"] + 1) ** 2
    params = 4 * (11 + 3 * hh)
    if what == "density":   # parameters and moments in and out, the statistics in
        return {"bytes": case["n"] * (2 * 3 * params * (1 + case["share"] / 2) + 8), "flops": 0}
    px, n = case["w"] * case["h"], case["n"]
    share, pairs = _pairs(case)
    kept = n * (4 * 11 + share * 12 * hh)   # the colours of what is in view only
    if what in ("render", "view"):
        return {"bytes": kept + px * (16 if what == "render" else 23), "flops": 21 * pairs + n * share * 500}
    if what == "grad":
        return {"bytes": kept + px * (16 + 4 + 12) + n * (4 + 36 + params),
                "flops": 81 * pairs + n * share * 2000}
    # a training step: parameters and moments in and out, the target in, the image out
    return {"bytes": n * 6 * params + 24 * px, "flops": 81 * pairs + n * share * 2000 + 3 * px * (8 * 44 + 60)}


def tolerance(case):
    what = case["what"]
    if what == "sort":
        return "exact"
    if what == "density":   # copies, but for the sampled positions of split Gaussians
        return {"rel": 1e-6, "max": 1e-5}
    if what == "loss":
        return {"rel": 1e-5, "max": 1e-3}
    # images: the forward pass is pinned bit for bit by the tests. (In 64 bits some pixels stop
    # one Gaussian earlier or later, which alone puts T 4e-3 away at a million Gaussians.)
    if what == "render":
        return {"rel": 1e-4, "max": 0.02}
    if what == "view":
        return {"rel": 1e-4, "max": 0.02, "differ": 1e-4}
    # gradients: 2e-4 from 64 bits, largest differences 2.5e-2 of the root mean square
    if what == "grad":
        return {"rel": 1e-3, "max": 0.1, "differ": 1e-4}
    return {"rel": 2e-3, "max": 0.2}   # moments: 5e-4 from 64 bits


# ------------------------------------------------------------------------------------
# The same in 64 bits
# ------------------------------------------------------------------------------------

C0, C1 = 0.28209479177387814, 0.4886025119029199
C2 = (1.0925484305920792, 0.31539156525252005, 0.5462742152960396)
C3 = (0.5900435899266435, 2.890611442640554, 0.4570457994644658, 0.3731763325901154, 1.445305721320277)


def _rotation(q):
    q = q / q.norm(dim=1, keepdim=True)
    r, x, y, z = q.unbind(1)
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - r * z), 2 * (x * z + r * y),
                        2 * (x * y + r * z), 1 - 2 * (x * x + z * z), 2 * (y * z - r * x),
                        2 * (x * z - r * y), 2 * (y * z + r * x), 1 - 2 * (x * x + y * y)], dim=1).reshape(-1, 3, 3)


def _basis(d, degree):
    x, y, z = d.unbind(1)
    b = [torch.full_like(x, C0)]
    if degree >= 1:
        b += [-C1 * y, C1 * z, -C1 * x]
    if degree >= 2:
        b += [C2[0] * x * y, -C2[0] * y * z, C2[1] * (2 * z * z - x * x - y * y), -C2[0] * x * z,
              C2[2] * (x * x - y * y)]
    if degree >= 3:
        b += [-C3[0] * y * (3 * x * x - y * y), C3[1] * x * y * z, -C3[2] * y * (4 * z * z - x * x - y * y),
              C3[3] * z * (2 * z * z - 3 * x * x - 3 * y * y), -C3[2] * x * (4 * z * z - x * x - y * y),
              C3[4] * z * (x * x - y * y), -C3[0] * x * (x * x - 3 * y * y)]
    return torch.stack(b, dim=1)


def _as(value, slope):
    """value, differentiated as slope."""
    return value.detach() + (slope - slope.detach())


def _records(mean, a, cov, sh, cam, o, degree):
    """Each Gaussian's [mu, a, conic, rgb] with the gradients of the reference's backward pass,
    its depth and its 2D covariance. cov is the 3D covariance (n, 3, 3), a the opacity."""
    P = torch.tensor(list(cam.P), dtype=torch.float64, device=DEV).reshape(3, 4)
    hom = mean @ P[:, :3].T + P[:, 3]
    r = hom[:, 2]
    mu = hom[:, :2] / r[:, None]
    lo = torch.tensor([o.clip_x_min, o.clip_y_min], dtype=torch.float64, device=DEV)
    hi = torch.tensor([o.clip_x_max, o.clip_y_max], dtype=torch.float64, device=DEV)
    rows = []
    for k in range(2):
        if o.clip_mode == abi.TDGS_CLIP_CLAMP:
            m = mu[:, k].detach().clamp(lo[k], hi[k])
            # inside, and at the upper bound, the clamped mean moves with the Gaussian; at the
            # lower one the reference's derivative carries 2 mu where the product rule gives mu
            moving = (hom[:, k] - hom[:, k].detach() + m * r.detach()) / r
            inside = (P[k, :3] - moving[:, None] * P[2, :3]) / r[:, None]
            fixed = (P[k, :3] - m[:, None] * P[2, :3]) / r[:, None]
            slope = (P[k, :3] - 2 * m[:, None] * P[2, :3]) / r[:, None]
            rows.append(torch.where((lo[k] < m)[:, None], inside, _as(fixed, slope)))
        else:
            rows.append((P[k, :3] - mu[:, k:k + 1] * P[2, :3]) / r[:, None])
    J = torch.stack(rows, dim=1)
    S = J @ cov @ J.transpose(1, 2)
    s11, s21, s22 = S[:, 0, 0], S[:, 1, 0], S[:, 1, 1]
    det0 = s11 * s22 - s21 * s21
    s11, s22 = s11 + o.dilation_x, s22 + o.dilation_y
    det = s11 * s22 - s21 * s21
    if o.antialiasing:   # the reference's gradient is that of the squared factor
        f = (det0.clamp(min=0) / det).sqrt().clamp(min=o.aa_min_factor).detach()
        a = a * f + a.detach() * (det0 / det - (det0 / det).detach())
    d = mean - torch.tensor(list(cam.position), dtype=torch.float64, device=DEV)
    d = d / d.norm(dim=1, keepdim=True)
    raw = torch.einsum("nk,nck->nc", _basis(d.detach(), degree), sh) + 0.5
    swapped = sh.detach()
    if degree == 3:   # the reference's direction Jacobian reads coefficient 15 for basis 16
        swapped = torch.cat([swapped[:, :, :15], swapped[:, :, 14:15]], dim=2)
    along = torch.einsum("nk,nck->nc", _basis(d, degree), swapped)
    along = torch.where(raw.detach() > 0, along, along.detach())
    rgb = raw.detach().clamp(min=0) + (raw - raw.detach()) + (along - along.detach())
    rec = torch.cat([mu, a[:, None], (s22 / det)[:, None], (-s21 / det)[:, None], (s11 / det)[:, None], rgb], dim=1)
    return rec, r, s11.detach(), s22.detach()


def _keep(mean, a, cam, o):
    P = torch.tensor(list(cam.P), dtype=torch.float64, device=DEV).reshape(3, 4)
    hom = mean @ P[:, :3].T + P[:, 3]
    r = hom[:, 2]
    keep = (a >= o.min_alpha) & (r > cam.near_z) & (r <= cam.far_z)
    if o.clip_mode == abi.TDGS_CLIP_FILTER:
        u, v = hom[:, 0] / r, hom[:, 1] / r
        keep &= (o.clip_x_min < u) & (u <= o.clip_x_max) & (o.clip_y_min < v) & (v <= o.clip_y_max)
    return keep.nonzero()[:, 0]


def _tiles(rec, r, s11, s22, case, o):
    """The tiles' lists in depth order: Gaussian of each entry, and where each tile's entries start."""
    w, h, tw, th = case["w"], case["h"], case["tw"], case["th"]
    a = rec[:, 2]
    gamma = 2 * (a / o.min_alpha).clamp(min=1e-30).log()
    rx, ry = (gamma.clamp(min=0) * s11).sqrt(), (gamma.clamp(min=0) * s22).sqrt()
    left = (rec[:, 0] - rx + 0.5).ceil().clamp(1, w + 1)
    top = (rec[:, 1] - ry + 0.5).ceil().clamp(1, h + 1)
    right = (rec[:, 0] + rx).round().clamp(0, w)
    bottom = (rec[:, 1] + ry).round().clamp(0, h)
    ok = (a >= o.min_alpha) & (left <= right) & (top <= bottom)
    tx0, tx1 = ((left - 1) / tw).floor().long(), ((right - 1) / tw).floor().long()
    ty0, ty1 = ((top - 1) / th).floor().long(), ((bottom - 1) / th).floor().long()
    ntx, nty = -(-w // tw), -(-h // th)
    order = torch.argsort(r, stable=True)
    order = order[ok[order]]
    cx, cy = (tx1 - tx0 + 1)[order], (ty1 - ty0 + 1)[order]
    count = cx * cy
    who = torch.repeat_interleave(torch.arange(order.numel(), device=DEV), count)
    k = torch.arange(who.numel(), device=DEV) - (count.cumsum(0) - count)[who]
    tile = (ty0[order][who] + k // cx[who]) * ntx + tx0[order][who] + k % cx[who]
    by_tile = torch.argsort(tile, stable=True)
    sizes = torch.bincount(tile, minlength=ntx * nty)
    return order[who[by_tile]], sizes, sizes.cumsum(0) - sizes, ntx


def _blend(rec, depth, lists, case, o, rgb_grad=None):
    """rgb, T and depth images, and with rgb_grad the gradient of rec."""
    entries, sizes, starts, ntx = lists
    w, h, tw, th = case["w"], case["h"], case["tw"], case["th"]
    bg = torch.tensor(list(o.background), dtype=torch.float64, device=DEV)
    rgb = bg.expand(w, h, 3).clone()
    T_img = torch.ones((w, h), dtype=torch.float64, device=DEV)
    D_img = torch.zeros((w, h), dtype=torch.float64, device=DEV)
    rec = rec.detach()
    grad = torch.zeros_like(rec) if rgb_grad is not None else None
    by_size = torch.argsort(sizes, descending=True)
    lens = sizes[by_size].tolist()
    px = torch.arange(tw * th, device=DEV)
    at = 0
    while at < len(lens) and lens[at] > 0:
        longest = lens[at]
        count = max(1, int(1.6e7 // (longest * tw * th)))
        t = by_size[at:at + count]
        at += count
        k = torch.arange(longest, device=DEV)
        valid = k[None, :] < sizes[t][:, None]
        idx = entries[(starts[t][:, None] + k).clamp(max=entries.numel() - 1)]
        U = (t % ntx)[:, None] * tw + px // th
        V = (t // ntx)[:, None] * th + px % th
        on = (U < w) & (V < h)
        R = rec[idx].requires_grad_(rgb_grad is not None)             # (tiles, entries, 9)
        cu, cv = U.double() + 0.5, V.double() + 0.5
        du = cu[:, None, :] - R[:, :, 0:1]
        dv = cv[:, None, :] - R[:, :, 1:2]
        e = -0.5 * (R[:, :, 3:4] * du * du + R[:, :, 5:6] * dv * dv) - R[:, :, 4:5] * du * dv
        with torch.no_grad():
            G = e.exp()
            al = (R[:, :, 2:3] * G).clamp(max=o.max_alpha)
            hit = (al >= o.min_alpha) & valid[:, :, None]
            al = torch.where(hit, al, 0.0)
            Tn = torch.cumprod(1 - al, dim=1)
            hit &= Tn >= o.min_transmittance
            al = torch.where(hit, al, 0.0)
            del Tn
        if rgb_grad is not None:   # d alpha: alpha along the exponent and G along the opacity
            al = al + torch.where(hit, al * (e - e.detach()) + G * (R[:, :, 2:3] - R[:, :, 2:3].detach()), 0.0)
        T = torch.cumprod(1 - al, dim=1)
        wt = al * torch.cat([torch.ones_like(T[:, :1]), T[:, :-1]], dim=1)
        C = torch.bmm(wt.transpose(1, 2).contiguous(), R[:, :, 6:9].contiguous()) + T[:, -1, :, None] * bg
        u, v = U[on], V[on]
        with torch.no_grad():
            rgb[u, v] = C[on]
            T_img[u, v] = T[:, -1][on]
            D_img[u, v] = torch.bmm(depth[idx][:, None, :], wt)[:, 0][on]
        if rgb_grad is not None:
            g, = torch.autograd.grad(C[on], R, rgb_grad[u, v])
            grad.index_add_(0, idx.reshape(-1), torch.where(valid[:, :, None], g, 0.0).reshape(-1, 9))
    return rgb, T_img, D_img, grad


def _filter(x, dim):
    """11 taps of a Gaussian of sigma 1.5 along dim, zeros outside."""
    wt = [math.exp(-(k * k) / 4.5) for k in range(-5, 6)]
    pad = [0, 0] * (x.dim() - 1 - dim) + [5, 5]
    xp = torch.nn.functional.pad(x, pad)
    return sum(wt[k] / sum(wt) * xp.narrow(dim, k, x.shape[dim]) for k in range(11))


def _loss(rgb, gt, weight):
    """The gradient of the training loss by rgb, and its two sums."""
    K = rgb.detach().requires_grad_(True)
    n = K.numel()
    mu1, mu2 = _filter(_filter(K, 0), 1), _filter(_filter(gt, 0), 1)
    s1 = _filter(_filter(K * K, 0), 1) - mu1 * mu1
    s2 = _filter(_filter(gt * gt, 0), 1) - mu2 * mu2
    s12 = _filter(_filter(K * gt, 0), 1) - mu1 * mu2
    ssim = ((2 * mu1 * mu2 + 1e-4) * (2 * s12 + 9e-4)) / ((mu1 * mu1 + mu2 * mu2 + 1e-4) * (s1 + s2 + 9e-4))
    g, = torch.autograd.grad(ssim.sum(), K)
    with torch.no_grad():
        grad = (1 - weight) / n * torch.where(K > gt, 1.0, -1.0) - weight / n * g
        return grad, torch.stack([(K - gt).abs().sum(), ssim.sum()])


def _render64(case, seed, cam, options, rgb_grad=None):
    """The render of a case and, for an image gradient (a tensor, or a function of the image),
    the gradients of records and parameters of the kept Gaussians."""
    o, c = options.to_c(), cam.to_c()
    mo, scaling, q, sh = (t.double() for t in _scene(case, seed))
    keep = _keep(mo[:, :3], torch.sigmoid(mo[:, 3]), c, o)
    leaves = [t[keep].requires_grad_(rgb_grad is not None) for t in (mo[:, :3], mo[:, 3], scaling, q, sh)]
    mean, logit, ls, qq, shk = leaves
    M = _rotation(qq) * ls.exp()[:, None, :]
    rec, depth, s11, s22 = _records(mean, torch.sigmoid(logit), M @ M.transpose(1, 2), shk, c, o, case["degree"])
    with torch.no_grad():
        lists = _tiles(rec.detach(), depth.detach(), s11, s22, case, o)
    image = None
    if callable(rgb_grad):
        image = _blend(rec, depth.detach(), lists, case, o)[0]
        rgb_grad = rgb_grad(image)
    rgb, T, D, g2 = _blend(rec, depth.detach(), lists, case, o, rgb_grad)
    out = {"rgb": rgb, "T": T, "depth": D, "gidx": keep, "rgb_grad": rgb_grad}
    if g2 is not None:
        listed_ = torch.zeros(keep.numel(), dtype=torch.bool, device=DEV)
        listed_[lists[0]] = True
        grads = torch.autograd.grad(rec, leaves, g2)
        out["g2"] = g2
        out["g3"] = [torch.where(listed_.reshape(-1, *[1] * (x.dim() - 1)), x, 0.0) for x in grads]
    return out


def exact(case, seed):
    what = case["what"]
    if what in ("sort", "density"):
        return None
    if what == "loss":
        gt = _image(case, seed + 1)
        rgb = (0.7 * gt + 0.3 * _image(case, seed)).double()
        grad, sums = _loss(rgb, gt.double(), case["weight"])
        return {"grad": grad, "sums": sums}
    if case["scene"] == "dense":   # minutes in 64 bits
        return None
    cam = _camera(case, seed)
    options = _options(case, cam)
    if what in ("render", "view"):
        r = _render64(case, seed, cam, options)
        if what == "render":
            return {"rgb": r["rgb"], "T": r["T"]}
        return {"rgb": r["rgb"], "T": r["T"], "depth": r["depth"], "image": None}
    if what == "grad":
        r = _render64(case, seed, cam, options, _image_grad(case, seed).double())
        g2, mean, logit, ls, q, sh = (torch.cat([x, x.new_zeros(case["n"] - x.shape[0], *x.shape[1:])])
                                      for x in [r["g2"]] + r["g3"])
        return {"rgb": r["rgb"], "T": r["T"], "last": None, "kept": None, "mean2d": g2[:, :2],
                "opacity2d": g2[:, 2], "conic": g2[:, 3:6], "color": g2[:, 6:9], "mean": mean, "opacity": logit,
                "scaling": ls, "rotation": q, "sh": sh}
    # a training step: the first camera of the trainer's seeded order
    k = int(np.random.Generator(np.random.PCG64(int(seed) & 0xffff)).permutation(4)[0])
    gt = _image(case, 4 * seed + k).double()
    sums = []

    def loss_grad(image):
        g, s = _loss(image, gt, WEIGHT)
        sums.append(s)
        return g

    r = _render64(case, seed, _camera(case, seed, k), options, loss_grad)
    p = [t.double() for t in _scene(case, seed)]
    mo, scaling, q, sh = p
    m = {k: v.double() for k, v in _moments(case, seed, case["n"], sh.shape[2]).items()}
    opt, keep, t = _training_options(case), r["gidx"], UPDATES + 1
    g = r["g3"]
    b1, b2 = float(np.float32(training.DEFAULT_BETA1)), float(np.float32(training.DEFAULT_BETA2))

    def adam(x, mom, grad, lr):
        m1 = b1 * mom[keep][..., 0] + (1 - b1) * grad
        m2 = b2 * mom[keep][..., 1] + (1 - b2) * grad * grad
        x[keep] -= lr * (m1 / (1 - b1 ** t)) / ((m2 / (1 - b2 ** t)).sqrt() + training.DEFAULT_EPSILON)
        mom[keep] = torch.stack([m1, m2], dim=-1)

    lr_sh = torch.full((sh.shape[2],), opt.sh_coeffs_rest_lr, dtype=torch.float64, device=DEV)
    lr_sh[0] = opt.sh_coeffs_dc_lr
    mean, logit = mo[:, :3].clone(), mo[:, 3].clone()
    adam(mean, m["means"], g[0], opt.initial_means_lr)
    adam(logit, m["opacity"], g[1], opt.opacity_features_lr)
    adam(scaling, m["scaling"], g[2], opt.scaling_features_lr)
    adam(q, m["rotation"], g[3], opt.rotation_features_lr)
    adam(sh, m["sh"], g[4], lr_sh)
    return {"rgb": r["rgb"], "loss_sums": sums[0], "rgb_grad": r["rgb_grad"],
            "means_opacity": torch.cat([mean, logit[:, None]], dim=1), "scaling": scaling, "rotation": q, "sh": sh,
            "m_means": m["means"], "m_opacity": m["opacity"], "m_scaling": m["scaling"], "m_rotation": m["rotation"],
            "m_sh": m["sh"]}
