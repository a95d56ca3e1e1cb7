"""Performance cases of the renderer and its denoisers: what a program that uses this package runs, through the
public entry points of cloudrendering_amd.vpt and cloudrendering_amd.kpn.

A case is a dict of plain values; its "kind" selects the path:

  frame          vpt.render_frame of one view: `mode` over the volume `volume`, width x height x spp
  inputs         kpn.render_inputs: the same with the feature maps the kernel-prediction denoiser reads
  eaw            a low-sample frame filtered by the edge-avoiding a-trous denoiser inside render_frame
  svgf           a clip of one-sample frames with a moving camera through the temporal denoiser
  batch          vpt.batch_render of a queue of requests over several volumes
  transmittance  vpt.transmittance_batch over a list of rays
  denoise        KpnDenoiser.denoise of a frame or of crops
  train          KpnDenoiser.train_step on a batch of crops, with the gradients read back
  pixel_kernel   vpt.per_pixel_kernel_forward
  inv_iter       vpt.inv_iter_kernel (blend, softmax and 5x5 kernel of one inverse iteration)

The renderer, its volume, the batched queue and the network are one per process, so the volume, the queue and the
network's weights belong to a case, and a seed selects what changes from call to call: the camera, the sample seeds,
the rays, the images. Volumes are the seeded fBm clouds of the benchmark and the tests.
"""
import math

import numpy as np
import torch

from cloudrendering_amd import kpn, vpt

# name: (sparse, edge, fBm seed). Dense: smoothstep(0.45, 0.6), about 30 % nonzero; sparse: smoothstep(0.645, 0.795),
# about 12 % active.
VOLUMES = {
    "dense64": (False, 64, 100),
    "dense128": (False, 128, 1),
    "dense256": (False, 256, 102),
    "sparse256": (True, 256, 7),
    "sparse512": (True, 512, 0),
}
# vpt mode number: (density and table bytes a path reads on average, floating-point and integer operations of its
# walker steps), counted by the work counters on the 512^3 sparse and 128^3 dense clouds. One step needs a Philox block
# (10 rounds) and about 60 operations of cell walking, tap addressing and collision decision.
PATH_WORK = {0: (120, 6.0e3), 1: (130, 7.0e3), 2: (250, 1.2e4), 3: (120, 6.0e3), 4: (1000, 6.0e4), 5: (4600, 2.2e5),
             6: (4600, 2.4e5)}
TRANSMITTANCE = {"delta": (40, 2.0e3), "ratio": (160, 8.0e3), "residual_ratio": (160, 8.0e3),
                 "decomposition": (40, 2.0e3)}
CONV_FLOPS = 2 * 9 * (15 * 32 + 4 * 32 * 32 + 32 * 25)  # per pixel of the denoiser network's forward pass


def listed():
    return [
        # An interactive preview: the smallest frame, where launches and host work are what counts.
        {"name": "preview_64", "kind": "frame", "volume": "dense64", "mode": 0, "width": 64, "height": 64, "spp": 1,
         "g": 0.5},
        # The dense next-event workload (environment image and sun, 64 bounces) at the benchmark's size.
        {"name": "nee_dense128_256", "kind": "frame", "volume": "dense128", "mode": 5, "width": 256, "height": 256,
         "spp": 64, "g": 0.85},
        # Frames of the 512^3 NanoVDB cloud: the cheap analog estimator, and the headline's dominant one.
        {"name": "delta_sparse512_1024", "kind": "frame", "volume": "sparse512", "mode": 0, "width": 1024,
         "height": 1024, "spp": 16, "g": 0.85},
        {"name": "rrt_sparse512_1024", "kind": "frame", "volume": "sparse512", "mode": 4, "width": 1024,
         "height": 1024, "spp": 16, "g": 0.5},
        # The denoiser's input render of a production frame (8 samples with feature maps).
        {"name": "inputs_1080p", "kind": "inputs", "volume": "dense128", "mode": 0, "width": 1920, "height": 1080,
         "spp": 8, "g": 0.5},
        # A low-sample frame through the spatial denoiser, four iterations as in the equal-time comparison.
        {"name": "eaw_1024", "kind": "eaw", "volume": "dense128", "mode": 0, "width": 1024, "height": 1024, "spp": 4,
         "g": 0.5, "iterations": 4},
        # A clip of one-sample frames through the temporal denoiser.
        {"name": "svgf_720p", "kind": "svgf", "volume": "dense128", "mode": 0, "width": 1280, "height": 720,
         "frames": 4, "g": 0.5},
        # A queue of mixed requests in one launch.
        {"name": "batch_8", "kind": "batch", "requests": 8, "side": 320, "spp": 24, "queue": 3},
        # 10^6 transmittance queries through the 512^3 cloud.
        {"name": "rays_1m", "kind": "transmittance", "volume": "sparse512", "estimator": "ratio", "rays": 1000000,
         "samples": 1},
        # Inference on a production frame, one training step on 16 crops of 128^2.
        {"name": "denoise_1080p", "kind": "denoise", "n": 1, "width": 1920, "height": 1080},
        {"name": "train_16x128", "kind": "train", "n": 16, "width": 128, "height": 128},
        # One inverse iteration of the kernel-prediction apply at full resolution.
        {"name": "inv_iter_1024", "kind": "inv_iter", "channels": 3, "width": 1024, "height": 1024, "kernel": 5,
         "use_previous": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "inputs", "eaw", "svgf", "batch", "transmittance", "denoise", "denoise",
                       "train", "pixel_kernel", "inv_iter"])
    c = {"kind": kind}
    if kind in ("frame", "inputs", "eaw", "svgf"):
        c["volume"] = rng.choice(sorted(VOLUMES))
        c["mode"] = rng.choice([0, 1, 2, 3, 4, 5, 6]) if kind == "frame" else rng.choice([0, 3, 4, 5])
        c["width"], c["height"] = _log_int(rng, 48, 1920), _log_int(rng, 48, 1080)
        c["g"] = round(rng.uniform(0.0, 0.85), 3)
    if kind == "frame":
        c["spp"] = _log_int(rng, 1, 64)
    elif kind == "inputs":
        c["spp"] = _log_int(rng, 2, 16)
    elif kind == "eaw":
        c["spp"], c["iterations"] = _log_int(rng, 1, 8), rng.randint(1, 5)
    elif kind == "svgf":
        c["frames"] = rng.randint(2, 5)
    elif kind == "batch":
        c.update(requests=rng.randint(2, 12), side=_log_int(rng, 96, 400), spp=_log_int(rng, 4, 64),
                 queue=rng.randint(0, 999))
    elif kind == "transmittance":
        c.update(volume=rng.choice(sorted(VOLUMES)), estimator=rng.choice(sorted(TRANSMITTANCE)),
                 rays=_log_int(rng, 1000, 1000000), samples=_log_int(rng, 1, 64))
    elif kind in ("denoise", "train"):
        n = rng.choice([1, 1, 4, 16]) if kind == "denoise" else rng.choice([4, 8, 16])
        big = 1920 if n == 1 else 160
        c.update(n=n, width=_log_int(rng, 32, big), height=_log_int(rng, 32, min(big, 1080)))
    elif kind == "pixel_kernel":
        c.update(n=rng.choice([1, 2]), channels=rng.choice([1, 3, 4]), width=_log_int(rng, 64, 1920),
                 height=_log_int(rng, 64, 1080), kernel=rng.choice([3, 5]))
    else:
        c.update(channels=rng.choice([1, 3, 4]), width=_log_int(rng, 64, 1920), height=_log_int(rng, 64, 1080),
                 kernel=rng.choice([3, 5]), use_previous=rng.random() < 0.5)
    return c


def _cost(c):
    w = work(c)
    return max(w["bytes"], w["flops"] / 50)


def draw(rng):
    """A case of the listed ranges; no larger than the largest listed case of its kind's family."""
    limit = max(_cost(c) for c in listed())
    while True:
        c = _draw(rng)
        if _cost(c) <= limit:
            return c


# --------------------------------------------------------------------------------------------------------------------
# work
# --------------------------------------------------------------------------------------------------------------------
def _batch_requests(c):
    """The queue's requests: volume, image side and spp by request, around the case's own."""
    rng = np.random.default_rng(c["queue"])
    names = ["dense64", "dense128", "dense256", "sparse256"]
    out = []
    for k in range(c["requests"]):
        out.append({"volume": names[k % len(names)], "side": int(c["side"] * rng.uniform(0.5, 1.0)),
                    "spp": max(1, int(c["spp"] * rng.uniform(0.5, 1.0))), "index": k,
                    "camera": _orbit(rng.uniform(0.0, 2.0 * math.pi), rng.uniform(-0.4, 1.0), 0.8)})
    return sorted(out, key=lambda q: q["volume"])


def work(c):
    k = c["kind"]
    if k in ("frame", "inputs", "eaw", "svgf"):
        px = c["width"] * c["height"]
        paths = px * (c["frames"] if k == "svgf" else c["spp"])
        b, f = PATH_WORK[c["mode"]]
        bytes_, flops = paths * b + 16 * px, paths * f
        if k == "inputs":
            bytes_ += px * 4 * 18
        if k == "eaw":  # per iteration and tap: three four-component distances and exponentials
            flops += px * c["iterations"] * 25 * 45
            bytes_ += px * 16 * 5
        if k == "svgf":
            flops += px * c["frames"] * 6 * 25 * 30
            bytes_ += px * c["frames"] * 16 * 12
        return {"bytes": bytes_, "flops": flops}
    if k == "batch":
        paths = sum(q["side"] ** 2 * q["spp"] for q in _batch_requests(c))
        return {"bytes": paths * PATH_WORK[5][0], "flops": paths * PATH_WORK[5][1]}
    if k == "transmittance":
        b, f = TRANSMITTANCE[c["estimator"]]
        return {"bytes": c["rays"] * (32 + b * c["samples"]), "flops": c["rays"] * f * c["samples"]}
    if k in ("denoise", "train"):
        px = c["n"] * c["width"] * c["height"]
        io = 4 * (15 + 3 + 3)
        return {"bytes": px * io + 4 * kpn.NUM_PARAMS * (1 if k == "denoise" else 5),
                "flops": px * CONV_FLOPS * (1 if k == "denoise" else 3)}
    px, ch, kk = c["width"] * c["height"], c["channels"], c["kernel"] ** 2
    if k == "pixel_kernel":
        return {"bytes": 4 * c["n"] * px * (kk + 2 * ch), "flops": 2 * c["n"] * px * kk * ch}
    reads = kk + 3 + ch * (2 if c["use_previous"] else 1) + 0.5 * ch
    return {"bytes": 4 * px * (reads + ch), "flops": px * (2 * kk * ch + 4 * kk)}


# --------------------------------------------------------------------------------------------------------------------
# renderer state
# --------------------------------------------------------------------------------------------------------------------
_now = {"volume": None, "queue": None, "started": False}


def _start():
    if not _now["started"]:
        vpt.initialize()
        _now["started"] = True


def _volume(name):
    """Loads the named cloud unless it is the current volume."""
    if _now["volume"] == name:
        return
    sparse, n, seed = VOLUMES[name]
    e0, e1 = (0.645, 0.795) if sparse else (0.45, 0.6)
    vpt.generate_fbm_cloud(n, n, n, seed=seed, octaves=5, lacunarity=2.0, gain=0.5, base_frequency=4.0, edge0=e0,
                           edge1=e1)
    vpt.set_use_sparse_grid(sparse)
    vpt.set_super_voxel_size(16 if sparse else 8)
    _now["volume"] = name


def _settings(mode, g):
    """The medium and light of the benchmark workloads: extinction 1024, albedo 0.9, at most 128 bounces; next-event
    tracking with an environment image and a directional sun, the other estimators with the default sky."""
    vpt.set_denoiser("None")
    vpt.set_use_feature_maps([])
    vpt.set_launch_config(0, 0, 0)
    vpt.set_vpt_mode(mode)
    vpt.set_grid_interpolation_type(1)
    vpt.set_extinction_base([1.0, 1.0, 1.0] if mode not in (1, 6) else [1.0, 0.8, 0.6])
    vpt.set_extinction_scale(1024.0)
    vpt.set_scattering_albedo([0.9, 0.9, 0.9])
    vpt.set_phase_g(g)
    vpt.set_max_bounces(64 if mode in (5, 6) else 128)
    vpt.clear_lights()
    if mode in (5, 6):
        vpt.load_environment_map_from_tensor(torch.ones((3, 16, 32), dtype=torch.float32))
        vpt.set_use_lights(True)
        vpt.add_light()
        vpt.set_light_property(0, "type", "Directional Light")
        vpt.set_light_property(0, "space", "World")
        vpt.set_light_property(0, "position", "58.26 76.6 27.17")
        vpt.set_light_property(0, "color", "1 0.961538462 0.884615385")
        vpt.set_light_property(0, "intensity", "2.6")
    else:
        vpt.set_use_builtin_environment_map("Default")
        vpt.set_use_lights(False)


def _orbit(az, el, d):
    return [d * math.cos(el) * math.sin(az), d * math.sin(el), d * math.cos(el) * math.cos(az)]


def _queue(c):
    """Fills the batched queue with the case's requests unless it holds them."""
    key = tuple(sorted((k, v) for k, v in c.items() if k != "name"))
    if _now["queue"] == key:
        return
    vpt.batch_clear()
    vpt.set_denoiser("None")
    vpt.set_use_feature_maps([])
    _settings(5, 0.5)
    vpt.set_use_builtin_environment_map("Default")
    vpt.set_max_bounces(128)
    for q in _batch_requests(c):
        _volume(q["volume"])
        vpt.set_camera_position(q["camera"])
        vpt.set_camera_target([0.0, 0.0, 0.0])
        vpt.set_seed_offset(q["index"])
        vpt.batch_add_request(torch.zeros((3, q["side"], q["side"]), dtype=torch.float32, device="cuda"), q["spp"])
    vpt.batch_set_launch_config(0, 256, 16, 16)
    _now["queue"] = key


# --------------------------------------------------------------------------------------------------------------------
# denoiser inputs
# --------------------------------------------------------------------------------------------------------------------
def _smooth(gen, n, ch, h, w):
    """Smooth positive images: coarse uniform noise, bilinearly enlarged."""
    t = torch.rand((n, ch, max(2, h // 16), max(2, w // 16)), generator=gen, device="cuda")
    return torch.nn.functional.interpolate(t, size=(h, w), mode="bilinear", align_corners=False)


def _pair(gen, n, h, w, target):
    """Features [N, 15, H, W], noisy radiance and, for training, a target, distributed like kpn.render_inputs'."""
    clean = _smooth(gen, n, 3, h, w) ** 2 * 2.0
    noise = torch.empty((n, 3, h, w), device="cuda").exponential_(1.0, generator=gen)
    noisy = clean * noise
    f = torch.empty((n, 15, h, w), device="cuda")
    cover = _smooth(gen, n, 1, h, w)
    f[:, 0:3] = noisy
    f[:, 3:6] = 0.9 * cover
    f[:, 6:7] = 0.8 * cover
    f[:, 7:8] = 0.1 * cover
    f[:, 8:9] = 1.0 - cover
    f[:, 9:11] = torch.randn((n, 2, h, w), generator=gen, device="cuda")
    # where the averaged normal lies on a view axis the screen-space gradient is infinite, or no number
    at = torch.randint(0, h * w, (4,), generator=gen, device="cuda").tolist()
    g = f[:, 9].reshape(n, -1).clone()
    g[:, at[0]], g[:, at[1]], g[:, at[2]] = float("inf"), float("-inf"), float("nan")
    f[:, 9] = g.reshape(n, h, w)
    f[:, 11:14] = clean * clean
    f[:, 14:15] = cover * torch.rand((n, 1, h, w), generator=gen, device="cuda")
    return f.contiguous(), noisy.contiguous(), clean.contiguous() if target else None


def _network():
    """The weights of the denoiser network (He-uniform, zero padding channels) as the flat parameter vector."""
    rng = np.random.default_rng(12)
    wts = np.zeros((6, 32, 32, 3, 3), np.float32)
    bias = np.zeros((6, 32), np.float32)
    for layer in range(6):
        ci, co = (15 if layer == 0 else 32), (25 if layer == 5 else 32)
        wts[layer, :co, :ci] = rng.uniform(-1.0, 1.0, (co, ci, 3, 3)) * math.sqrt(6.0 / (9 * ci))
        bias[layer, :co] = rng.uniform(-0.05, 0.05, co)
    return np.concatenate([wts.reshape(-1), bias.reshape(-1)])


def _apply_inputs(c, gen):
    n, ch, h, w, k = c.get("n", 1), c["channels"], c["height"], c["width"], c["kernel"]
    img = _smooth(gen, n, ch, h, w) * 2.0 * torch.rand((n, ch, h, w), generator=gen, device="cuda")
    if c["kind"] == "pixel_kernel":
        wt = torch.softmax(torch.randn((n, k * k, h, w), generator=gen, device="cuda"), 1)
        return {"image": img, "weights": wt}
    lh, lw = (h + 1) // 2, (w + 1) // 2
    low = _smooth(gen, n, ch, lh, lw)
    return {"image": img, "low_pred": low, "low_x": low * 1.1, "prev": _smooth(gen, n, ch, h, w) * 2.0,
            "weights": torch.randn((n, k * k + 3, h, w), generator=gen, device="cuda")}


def _rays(c, gen):
    """Rays from a sphere around the volume towards points inside it."""
    n = c["rays"]
    o = torch.randn((n, 3), generator=gen, device="cuda")
    o = 0.8 * o / o.norm(dim=1, keepdim=True)
    to = (torch.rand((n, 3), generator=gen, device="cuda") - 0.5) * 0.4
    d = to - o
    return o.contiguous(), (d / d.norm(dim=1, keepdim=True)).contiguous()


# --------------------------------------------------------------------------------------------------------------------
# prepare and run
# --------------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    _start()
    c = dict(case)
    k = c["kind"]
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    s = {"case": c}
    if k in ("frame", "inputs", "eaw", "svgf"):
        _volume(c["volume"])
        _settings(c["mode"], c["g"])
        s["probe"] = torch.zeros((3, c["height"], c["width"]), dtype=torch.float32, device="cuda")
        az, el, d = rng.uniform(0.0, 2.0 * math.pi), rng.uniform(-0.4, 1.0), rng.uniform(0.6, 0.8)
        s["cameras"] = [_orbit(az + 0.01 * f, el, d) for f in range(c.get("frames", 1))]
        s["seed"] = int(rng.integers(1 << 20))
        vpt.set_camera_target([0.0, 0.0, 0.0])
        vpt.set_camera_position(s["cameras"][0])
        vpt.render_frame(s["probe"], 1)  # the volume's tables are built with the first frame
        if k == "eaw":
            vpt.set_denoiser("EAW")
            vpt.set_denoiser_property("maxNumIterations", str(c["iterations"]))
    elif k == "batch":
        _queue(c)
        s["offset"] = int(rng.integers(1 << 16)) * 1024
        vpt.batch_render(s["offset"] + 512)  # the queue's launch graph is captured with the first pass
    elif k == "transmittance":
        _volume(c["volume"])
        _settings({"residual_ratio": 4, "decomposition": 3}.get(c["estimator"], 0), 0.5)
        s["o"], s["d"] = _rays(c, gen)
        s["seed"] = int(rng.integers(1 << 20))
        vpt.transmittance_batch(c["estimator"], s["o"][:64], s["d"][:64], None, 1, 1)
    elif k in ("denoise", "train"):
        s["net"] = kpn.KpnDenoiser(parameters=_network())
        s["features"], s["noisy"], s["target"] = _pair(gen, c["n"], c["height"], c["width"], k == "train")
    else:
        s.update(_apply_inputs(c, gen))
    return s


def _view(s, f=0):
    vpt.set_camera_position(s["cameras"][f])
    vpt.set_seed_offset(s["seed"] + f)


def run(s):
    c = s["case"]
    k = c["kind"]
    if k in ("frame", "eaw"):
        _view(s)
        return vpt.render_frame(s["probe"], c["spp"])
    if k == "inputs":
        _view(s)
        return list(kpn.render_inputs(vpt, c["height"], c["width"], c["spp"]))
    if k == "svgf":
        vpt.set_denoiser("SVGF")
        vpt.set_denoiser_property("maxNumIterations", "5")
        out = []
        for f in range(c["frames"]):
            _view(s, f)
            if f == 0:
                vpt.set_view_projection_matrix_as_previous()
            out.append(vpt.render_frame(s["probe"], 1))
            vpt.set_view_projection_matrix_as_previous()
        return out
    if k == "batch":
        return vpt.batch_render(s["offset"])
    if k == "transmittance":
        return list(vpt.transmittance_batch(c["estimator"], s["o"], s["d"], None, c["samples"], s["seed"]))
    if k == "denoise":
        return s["net"].denoise(s["features"], s["noisy"])
    if k == "train":
        loss = s["net"].train_step(s["features"], s["noisy"], s["target"], 1e-3)
        return {"loss": loss, "gradients": s["net"].gradients()}
    if k == "pixel_kernel":
        return vpt.per_pixel_kernel_forward(s["image"], s["weights"], c["kernel"])
    return vpt.inv_iter_kernel(s["image"], s["low_pred"], s["low_x"], s["prev"] if c["use_previous"] else None,
                               s["weights"], c["kernel"], c["use_previous"])


# --------------------------------------------------------------------------------------------------------------------
# 64-bit values
# --------------------------------------------------------------------------------------------------------------------
def _shifted(img, dy, dx):
    """img[..., y + dy, x + dx], zero outside."""
    h, w = img.shape[-2:]
    r = max(abs(dy), abs(dx))
    p = torch.nn.functional.pad(img, (r, r, r, r))
    return p[..., r + dy:r + dy + h, r + dx:r + dx + w]


def _filter(image, weights, k):
    out = torch.zeros_like(image)
    for t in range(k * k):
        out = out + weights[:, t:t + 1] * _shifted(image, t // k - k // 2, t % k - k // 2)
    return out


def _forward64(wts, bias, features):
    """The network's logits [N, 25, H, W]: cleaned features, five ReLU layers and the linear one."""
    f = features.double()
    grad = torch.nan_to_num(f[:, 9:11], nan=0.0, posinf=16.0, neginf=-16.0).clamp(-16.0, 16.0)
    x = torch.where(torch.isfinite(f), f, torch.zeros_like(f))
    x = torch.cat([torch.log1p(x[:, 0:3].clamp(min=0.0)), x[:, 3:9], grad, torch.log1p(x[:, 11:14].clamp(min=0.0)),
                   x[:, 14:15]], 1)
    x = torch.nn.functional.pad(x, (0, 0, 0, 0, 0, 17))
    for layer in range(6):
        z = 0.0
        for t in range(9):
            z = z + torch.matmul(_shifted(x, t // 3 - 1, t % 3 - 1).movedim(1, -1), wts[layer][:, :, t // 3, t % 3].t())
        z = (z + bias[layer]).movedim(-1, 1)
        x = torch.relu(z) if layer < 5 else z
    return x[:, :25]


def exact(case, seed):
    """Monte Carlo renders have no 64-bit value; the network and the kernel-prediction apply have."""
    c = dict(case)
    k = c["kind"]
    if k in ("frame", "inputs", "eaw", "svgf", "batch", "transmittance"):
        return None
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    if k in ("denoise", "train"):
        f, noisy, target = _pair(gen, c["n"], c["height"], c["width"], k == "train")
        flat = torch.from_numpy(_network()).double().cuda()
        wts = flat[:6 * 9216].reshape(6, 32, 32, 3, 3).clone().requires_grad_(k == "train")
        bias = flat[6 * 9216:].reshape(6, 32).clone().requires_grad_(k == "train")
        out = _filter(noisy.double(), torch.softmax(_forward64(wts, bias, f), 1), 5)
        if k == "denoise":
            return out
        t = target.double()
        loss = (((out - t) ** 2) / (t * t + 0.01)).mean()
        loss.backward()
        g = torch.cat([wts.grad.reshape(-1), bias.grad.reshape(-1)]).cpu().numpy()
        return {"loss": float(loss.detach()), "gradients": g}
    s = {a: t.double() for a, t in _apply_inputs(c, gen).items()}
    if k == "pixel_kernel":
        return _filter(s["image"], s["weights"], c["kernel"])
    kk = c["kernel"] ** 2
    lf_w, hf_w, pr_w = (torch.sigmoid(s["weights"][:, kk + i:kk + i + 1]) for i in range(3))
    up = [t.repeat_interleave(2, 2).repeat_interleave(2, 3)[..., :c["height"], :c["width"]]
          for t in (s["low_pred"], s["low_x"])]
    lf = lf_w * up[0] + (1.0 - lf_w) * up[1]
    if c["use_previous"]:
        lf = lf * (1.0 - pr_w) + s["prev"] * pr_w
    base = hf_w * (s["image"] - up[1] + lf) + (1.0 - hf_w) * lf
    return _filter(base, torch.softmax(s["weights"][:, :kk], 1), c["kernel"])
