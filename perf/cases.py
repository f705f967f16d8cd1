"""Timed cases of the NCS noise correction on one MI355X.

Each case is one call (or one training step, or a few frames of a stream) as a
program that uses the package makes it, through the package's public entry
points.  Inputs are synthetic sCMOS scenes with the statistics of
ncs_amd/sim.py (worm-like filaments, Gaussian PSF, per-pixel gain, offset and
read variance), rendered on the GPU so that they are quick to make.

    listed()             the cases that are always timed
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what the program holds before the call
    run(state)           one pass; returns its outputs
    work(case)           bytes and flops that a pass cannot do without
    exact(case, seed)    the outputs in 64 bits, by plain torch

Outputs that the entry points give in 64-bit floats but compute in 32 (the C
library's whole-image call) are cast to float32, which is exact.
"""
import ctypes
import math

import numpy
import torch

from ncs_amd import _lib, linstart, masks, ncs, ncs_c, sim, warmstart

DEV = "cuda:0"


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # The smallest call in earnest: the correction of one region of
        # interest around a few molecules, from Python, as a script or a
        # viewer makes it.  30 windows: launches and host work.
        dict(name="roi_64x80", path="host", frames=1, height=64, width=80, alpha=0.1),
        # The demo of the reference's GPU hosts: a series of 50 small frames
        # in one call (one gamma map for all of them).
        dict(name="series_50x128x128", path="host", frames=50, height=128, width=128, alpha=0.1),
        # One ordinary camera region, odd and unequal sides, single call.
        dict(name="frame_501x643", path="host", frames=1, height=501, width=643, alpha=0.1),
        # The kernel batch interface on the inputs of the reference's own GPU
        # timing: 1000 independent 16 x 16 tiles, data U(10, 20), gamma
        # U(2, 4), Gaussian high-pass mask.
        dict(name="tiles_1000", path="tiles", tiles=1000, alpha=0.1),
        # A camera's time series: raw 16-bit frames in pinned host memory
        # through two captured pipelines, corrected frames back in host
        # memory, the host one frame ahead.
        dict(name="stream_4x2304_u16", path="stream", frames=4, height=2304, width=2304,
             alpha=0.1),
        # The batch of the benchmark: 10 frames of 2048 x 2048 resident on
        # the GPU, learned linear start, history 1, status and cost per tile.
        dict(name="batch_10x2048_linear", path="device", frames=10, height=2048, width=2048,
             start="linear", history=1, precision="fp32", mask="otf", alpha=0.1),
        # The same entry point with every parameter at its default (plain
        # start, history 5), as a first-time user of the device call has it.
        dict(name="batch_4x2048_default", path="device", frames=4, height=2048, width=2048,
             start="plain", history=5, precision="fp32", mask="otf", alpha=0.1),
        # The same entry point under an anisotropic mask (a microscope whose
        # OTF is not round), ragged sides.
        dict(name="batch_3x1000x1301_rotated", path="device", frames=3, height=1000, width=1301,
             start="plain", history=3, precision="fp32", mask="rotated", alpha=0.2),
        # The FP16-split option of the basis changes, which the caller picks.
        dict(name="batch_4x2048_f16split", path="device", frames=4, height=2048, width=2048,
             start="linear", history=1, precision="f16split", mask="otf", alpha=0.1),
        # Frames of many sizes and alphas in one launch (full frames, halves
        # and regions of interest of several fields of view): the uneven
        # batch of the benchmark in the reference tiling.
        dict(name="uneven_30", path="uneven", rois=16, small=8, half=4, full=2, layout=1),
        # The learned conv-net start in front of the solve.
        dict(name="learned_2x2048", path="device", frames=2, height=2048, width=2048,
             start="learned", history=5, precision="fp32", mask="otf", alpha=0.1),
        # One training step of the conv net (forward, loss, backward) at the
        # trainer's own batch size.
        dict(name="train_1024", path="train", tiles=1024),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "host", "tiles", "clib", "stream", "device", "device", "device",
                       "uneven", "train", "train"])
    if kind == "host":
        h, w = _log_int(rng, 30, 1100), _log_int(rng, 30, 1100)
        n = max(1, min(_log_int(rng, 1, 50), (1 << 20) // (h * w)))
        return dict(path="host", frames=n, height=h, width=w,
                    alpha=round(rng.uniform(0.05, 0.3), 3))
    if kind == "tiles":
        return dict(path="tiles", tiles=_log_int(rng, 50, 1000),
                    alpha=round(rng.uniform(0.05, 0.3), 3))
    if kind == "clib":
        # the C library's whole-image call: float64 in and out
        return dict(path="clib", height=_log_int(rng, 40, 400), width=_log_int(rng, 40, 400),
                    window=rng.choice([10, 12, 16]), alpha=round(rng.uniform(0.05, 0.3), 3))
    if kind == "stream":
        return dict(path="stream", frames=rng.randint(2, 6), height=_log_int(rng, 128, 2304),
                    width=_log_int(rng, 128, 2304), alpha=round(rng.uniform(0.05, 0.3), 3))
    if kind == "device":
        h, w = _log_int(rng, 200, 2304), _log_int(rng, 200, 2304)
        n = max(1, min(_log_int(rng, 1, 20), 10 * 2048 * 2048 // (h * w)))
        start = rng.choice(["plain", "linear", "linear", "learned"])
        if start == "learned":
            n = max(1, min(n, 2 * 2048 * 2048 // (h * w)))
        return dict(path="device", frames=n, height=h, width=w, start=start,
                    history=rng.choice([1, 2, 3, 5, 8]),
                    precision=rng.choice(["fp32", "fp32", "f16split"]),
                    mask=rng.choice(["otf", "otf", "rotated"]) if start == "plain" else "otf",
                    alpha=round(rng.uniform(0.05, 0.3), 3))
    if kind == "uneven":
        return dict(path="uneven", rois=rng.randint(2, 24), small=rng.randint(0, 8),
                    half=rng.randint(0, 4), full=rng.randint(0, 2), layout=rng.randint(2, 1 << 20))
    return dict(path="train", tiles=_log_int(rng, 100, 8000))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _uniform(shape, g, lo, hi, dtype=torch.float64):
    return torch.rand(shape, generator=g, device=DEV, dtype=dtype) * (hi - lo) + lo


def _filaments(h, w, g, background=20.0, photons_per_um=2000.0):
    """Ideal image of a worm-like-chain scene (sim.filament_scene on the GPU):
    emitters every 10 nm of filament, binned to pixels and blurred with the
    PSF."""
    n = max(1, int(round(sim.FILAMENTS_PER_UM2 * h * w * sim.PIXEL_UM ** 2)))
    m = 1500  # emitters of the longest filament (15 um)
    length = _uniform((n, 1), g, 500.0, 1500.0)
    theta = _uniform((n, 1), g, 0.0, 2.0 * math.pi) + torch.cumsum(
        torch.randn((n, m), generator=g, device=DEV, dtype=torch.float64) * 0.1, dim=1)
    row = _uniform((n, 1), g, 0.0, float(h)) + torch.cumsum(torch.cos(theta) * 0.1, dim=1)
    col = _uniform((n, 1), g, 0.0, float(w)) + torch.cumsum(torch.sin(theta) * 0.1, dim=1)
    ok = (torch.arange(m, device=DEV)[None, :] < length) & (row >= 0) & (row < h) & \
         (col >= 0) & (col < w)
    at = (row.floor() * w + col.floor()).long()[ok]
    img = torch.bincount(at, minlength=h * w).to(torch.float64).view(1, 1, h, w) * \
        (photons_per_um * 0.01)
    x = torch.arange(-4, 5, device=DEV, dtype=torch.float64)
    k = torch.exp(-0.5 * (x / sim.SIGMA_PX) ** 2)
    k = k / k.sum()
    pad = torch.nn.functional.pad(img, (4, 4, 4, 4), mode="replicate")
    # separable blur as shifted sums
    rows = sum(k[i] * pad[:, :, i:i + h, :] for i in range(9))
    out = sum(k[i] * rows[:, :, :, i:i + w] for i in range(9))
    return out.view(h, w) + background


def _camera(h, w, g, heavy_tail=False):
    offset = 100.0 + 2.0 * torch.randn((h, w), generator=g, device=DEV, dtype=torch.float64)
    gain = 2.0 + 0.2 * torch.randn((h, w), generator=g, device=DEV, dtype=torch.float64)
    gain = gain.clamp(min=1.0)
    var = (-50.0 * torch.log1p(-_uniform((h, w), g, 0.0, 1.0))).clamp(max=3000.0)
    if heavy_tail:
        hot = _uniform((h, w), g, 0.0, 1.0) < 0.01
        bright = torch.exp(7.0 + 0.5 * torch.randn((h, w), generator=g, device=DEV,
                                                   dtype=torch.float64))
        var = torch.where(hot, bright, var)
    return offset, gain, var


def _frame(h, w, g, camera):
    """Photo-electron image (float32, device) of one scene."""
    offset, gain, var = camera
    ideal = _filaments(h, w, g)
    adu = gain * torch.poisson(ideal, generator=g) + offset + torch.sqrt(var) * torch.randn(
        (h, w), generator=g, device=DEV, dtype=torch.float64)
    d = (adu - offset) / gain
    return torch.where(d <= 0, torch.full_like(d, 1.0e-6), d).float().contiguous()


def _mask(kind):
    """Centred 16 x 16 mask."""
    if kind == "otf":
        return masks.otf_mask()
    if kind == "gauss":
        return masks.gaussian_highpass_mask()
    # an anisotropic Gaussian high-pass, rotated; exactly point-symmetric
    k = numpy.fft.fftfreq(16, 1.0 / 16)
    ky, kx = numpy.meshgrid(k, k, indexing="ij")
    a = math.cos(0.5) * kx + math.sin(0.5) * ky
    b = -math.sin(0.5) * kx + math.cos(0.5) * ky
    m = 1.0 - numpy.exp(-(a / 3.0) ** 2 - (b / 6.0) ** 2)
    neg = (-numpy.arange(16)) % 16
    return numpy.fft.fftshift(0.5 * (m + m[neg][:, neg]))


def _same_size(case, seed):
    """(frames, one gamma map) of a batch of equal frames, on the device."""
    g = _generator(seed)
    h, w = case["height"], case["width"]
    camera = _camera(h, w, g)
    gamma = (camera[2] / camera[1] ** 2).float().contiguous()
    return [_frame(h, w, g, camera) for _ in range(case.get("frames", 1))], gamma


def _uneven_shapes(case):
    rng = numpy.random.default_rng(case["layout"])
    shapes = [(512, 512)] * case["small"] + [(1024, 2048)] * case["half"] + \
        [(2304, 2304)] * case["full"]
    shapes += [tuple(int(v) for v in rng.integers(64, 401, 2)) for _ in range(case["rois"])]
    alphas = [float(a) for a in rng.uniform(0.05, 0.3, len(shapes))]
    return shapes, alphas


def _uneven(case, seed):
    g = _generator(seed)
    shapes, alphas = _uneven_shapes(case)
    data, gamma = [], []
    for h, w in shapes:
        camera = _camera(h, w, g, heavy_tail=True)
        gamma.append((camera[2] / camera[1] ** 2).float().contiguous())
        data.append(_frame(h, w, g, camera))
    return data, gamma, shapes, alphas


def _raw_series(case, seed):
    """Raw uint16 frames (int32, device) of one camera, its maps in float32."""
    g = _generator(seed)
    h, w = case["height"], case["width"]
    maps = [m.float().double() for m in _camera(h, w, g)]
    offset, gain, var = maps
    raw = []
    for _ in range(case["frames"]):
        adu = gain * torch.poisson(_filaments(h, w, g), generator=g) + offset + \
            torch.sqrt(var) * torch.randn((h, w), generator=g, device=DEV, dtype=torch.float64)
        raw.append(torch.clamp(torch.round(adu), 0, 65535).to(torch.int32))
    return raw, offset, gain, var


def _tiles(case, seed):
    g = _generator(seed)
    n = case["tiles"]
    data = _uniform((n, 16, 16), g, 10.0, 20.0).float()
    gamma = _uniform((1, 16, 16), g, 2.0, 4.0).float().expand(n, 16, 16).contiguous()
    return data, gamma


def _train_inputs(case, seed):
    """Normalised tiles, a target correction and the parameters, on the
    device: tiles cut from a filament scene, the target a smoothed tile."""
    g = _generator(seed)
    n = case["tiles"]
    side = max(64, 16 * int(math.ceil(math.sqrt(n))))
    camera = _camera(side, side, g)
    data = _frame(side, side, g, camera)
    gamma = (camera[2] / camera[1] ** 2).float()

    def cut(a):
        k = side // 16
        return a.view(k, 16, k, 16).permute(0, 2, 1, 3).reshape(-1, 16, 16)[:n].contiguous()

    d, gm = cut(data), cut(gamma)
    x, sigma = warmstart.normalize(d, gm)
    smooth = torch.nn.functional.avg_pool2d(d[:, None], 3, stride=1, padding=1,
                                            count_include_pad=False)[:, 0]
    target = ((smooth - d) / sigma).contiguous()
    params = torch.from_numpy(warmstart.init_params(int(seed) & 0xFFFF)).to(DEV)
    # biases as training leaves them: small, not zero
    bias = torch.zeros_like(params)
    for _, b, _, _ in warmstart.layer_slices():
        bias[b] = 0.05 * torch.randn(b.stop - b.start, generator=g, device=DEV)
    return x, target, (params + bias).contiguous()


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------

_STARTS = {"plain": _lib.START_PLAIN, "linear": _lib.START_LINEAR, "learned": _lib.START_LEARNED}


def _device_state(data, gamma, alphas, mask, params, status_and_cost=True):
    """A batch resident on the GPU, as a program that calls the device entry
    point holds it."""
    ctx = _lib.context(0)
    ctx.set_otf_mask(masks.to_fft_order(mask).astype(numpy.float32))
    if params.start == _lib.START_LINEAR:
        ctx.set_linear_start(linstart.load(), linstart.load_slope(), linstart.ALPHA_REF)
    if params.start == _lib.START_LEARNED:
        warmstart.set_context_weights(warmstart.load())
    out = [torch.empty_like(d) for d in data]
    frames = [dict(data=d.data_ptr(), gamma=g.data_ptr(), out=o.data_ptr(), height=d.shape[0],
                   width=d.shape[1], alpha=a)
              for d, g, o, a in zip(data, gamma, out, alphas)]
    total = sum(_lib.tile_count(d.shape[0], d.shape[1]) for d in data)
    status = torch.empty(total, dtype=torch.int32, device=DEV)
    cost = torch.empty(total, dtype=torch.float32, device=DEV)
    return dict(kind="device", ctx=ctx, frames=frames, params=params, keep=(data, gamma),
                out=out, status=status, cost=cost)


def _device_params(case):
    return _lib.default_params(
        start=_STARTS[case["start"]], history=case["history"],
        precision=_lib.PRECISION_F16_SPLIT if case["precision"] == "f16split"
        else _lib.PRECISION_FP32)


def prepare(case, seed):
    path = case["path"]
    if path == "host":
        data, gamma = _same_size(case, seed)
        return dict(kind="host", images=[d.cpu().numpy() for d in data],
                    gamma=gamma.cpu().numpy(), mask=_mask("otf"), alpha=case["alpha"])
    if path == "clib":
        data, gamma = _same_size(case, seed)
        mask = masks.otf_mask(r=case["window"])
        return dict(kind="clib", image=data[0].double().cpu().numpy(),
                    gamma=gamma.double().cpu().numpy(), alpha=case["alpha"],
                    mask=numpy.ascontiguousarray(masks.to_fft_order(mask)))
    if path == "tiles":
        data, gamma = _tiles(case, seed)
        return dict(kind="tiles", data=data.cpu().numpy(), gamma=gamma.cpu().numpy(),
                    mask=masks.to_fft_order(_mask("gauss")), alpha=case["alpha"])
    if path == "device":
        data, gamma = _same_size(case, seed)
        return _device_state(data, [gamma] * len(data), [case["alpha"]] * len(data),
                             _mask(case["mask"]), _device_params(case))
    if path == "uneven":
        data, gamma, _, alphas = _uneven(case, seed)
        params = _lib.default_params(start=_lib.START_LINEAR, history=1)
        return _device_state(data, gamma, alphas, _mask("otf"), params)
    if path == "stream":
        raw, *maps = _raw_series(case, seed)
        ctx = _lib.context(0)
        ctx.set_otf_mask(masks.to_fft_order(_mask("otf")).astype(numpy.float32))
        shape = (case["height"], case["width"])
        maps = [m.float().cpu().numpy() for m in maps]
        lines = []
        for _ in range(2):
            pl = _lib.Pipeline(ctx, [shape], [case["alpha"]], input_format=_lib.INPUT_ADU_U16)
            pl.set_camera(0, *maps)
            lines.append(pl)
        ins, outs = [], []
        for r in raw:
            pin = torch.empty(shape, dtype=torch.int16, pin_memory=True)
            pin.numpy().view(numpy.uint16)[:] = r.cpu().numpy().astype(numpy.uint16)
            ins.append(pin)
            outs.append(torch.empty(shape, dtype=torch.float32, pin_memory=True))
        return dict(kind="stream", lines=lines, keep=(ins, outs),
                    ins=[a.numpy().view(numpy.uint16) for a in ins],
                    outs=[a.numpy() for a in outs])
    if path == "train":
        x, target, params = _train_inputs(case, seed)
        return dict(kind="train", x=x, target=target, params=params.requires_grad_(True))
    raise ValueError(path)


def run(state):
    kind = state["kind"]
    if kind == "host":
        return ncs.reduceNoise(state["images"], state["gamma"], state["mask"], state["alpha"])
    if kind == "clib":
        out = ncs_c.cReduceNoise(state["image"], state["gamma"], state["mask"], state["alpha"])
        return out.astype(numpy.float32)
    if kind == "tiles":
        u, _, status, cost = ncs.solveTiles(state["data"], state["gamma"], state["mask"],
                                            state["alpha"])
        return dict(u=u, status=status, cost=cost)
    if kind == "device":
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        state["ctx"].reduce_frames_device(state["frames"], state["params"],
                                          status_ptr=state["status"].data_ptr(),
                                          cost_ptr=state["cost"].data_ptr(), stream_ptr=stream)
        return dict(out=state["out"], status=state["status"], cost=state["cost"])
    if kind == "stream":
        lines, last = state["lines"], None
        for k, (raw, out) in enumerate(zip(state["ins"], state["outs"])):
            pl = lines[k % 2]
            seq = pl.launch([raw], [out])
            if last is not None:  # the frame before this one is used now
                last[0].wait(last[1])
            last = (pl, seq)
        last[0].wait(last[1])
        return state["outs"]
    # one training step up to the gradients, as warmstart.train makes it
    p = state["params"]
    p.grad = None
    y = warmstart.NetFunction.apply(p, state["x"])
    loss = torch.mean((y - state["target"]) ** 2)
    loss.backward()
    return dict(y=y.detach(), loss=loss.detach(), grad=p.grad)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

_NET_MACS = 256 * 9 * (2 * 32 + 32 * 32 + 32 * 32 + 32)  # one tile, forward


def _solve_flops(pixels, owned):
    """A solve needs at least two iterations of two 16 x 16 basis changes
    (2 x 16^3 multiply-adds each) and about 60 operations per pixel, on the
    256 pixels of each tile, which owns `owned` of them."""
    return pixels / float(owned) * 2 * (2 * 2 * 2 * 4096 + 60 * 256)


def work(case):
    path = case["path"]
    if path == "train":
        n = case["tiles"]
        # inputs, target and output once, the three saved activations written
        # and read (BF16), parameters and gradients; forward, data gradient
        # of layers 2-4 and weight gradients of all four
        back = 256 * 9 * (32 * 32 + 32 * 32 + 32)
        return dict(bytes=n * (2048 + 2 * 1024 + 2 * 3 * 256 * 32 * 2) + 2 * 4 * 19393,
                    flops=2.0 * n * (2 * _NET_MACS + back))
    if path == "uneven":
        shapes, _ = _uneven_shapes(case)
    elif path == "tiles":
        shapes = [(16 * case["tiles"], 16)]
    else:
        shapes = [(case["height"], case["width"])] * case.get("frames", 1)
    pixels = sum(h * w for h, w in shapes)
    shared_gamma = path in ("host", "device", "clib")
    gamma_pixels = shapes[0][0] * shapes[0][1] if shared_gamma else pixels
    size = 8 if path == "clib" else 4
    if path == "stream":  # raw frames and three maps in, images out
        return dict(bytes=pixels * 6 + 12 * pixels // len(shapes), flops=_solve_flops(pixels, 196))
    owned = 256 if path == "tiles" else 196
    flops = _solve_flops(pixels, owned)
    if case.get("start") == "learned":
        flops += pixels / 196.0 * 2 * _NET_MACS
    # data and gamma in, image out
    return dict(bytes=size * (2 * pixels + gamma_pixels), flops=flops)


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _minimise(d, g, mask_fft, alpha):
    """Minimiser of sum(u - (d + g) ln(u + g)) + alpha / r^2 sum(q |FFT u|^2)
    for tiles [n, r, r] in float64 (damped Newton steps, each solved by
    preconditioned conjugate gradients), and its cost per tile.  The
    likelihood is a barrier at u + g = 0, so the guard at 1e-6 plays no part
    at the minimiser."""
    n, r, _ = d.shape
    m = torch.from_numpy(numpy.asarray(mask_fft, dtype=numpy.float32)).to(DEV).double()
    q = m * m
    flip = (-torch.arange(r, device=DEV)) % r
    q = 0.5 * (q + q[flip][:, flip])
    a = torch.as_tensor(alpha, dtype=torch.float64, device=DEV).reshape(-1, 1, 1)
    c = d + g

    def k_of(x):  # gradient of the noise term, without alpha
        return torch.fft.ifft2(2.0 * q * torch.fft.fft2(x)).real

    def dot(x, y):
        return (x * y).sum(dim=(1, 2), keepdim=True)

    def cost_of(x):
        nc = (q * torch.fft.fft2(x).abs() ** 2).sum(dim=(1, 2), keepdim=True) / (r * r)
        return (x - c * torch.log(x + g)).sum(dim=(1, 2), keepdim=True) + a * nc

    u = d.clone()
    for _ in range(40):
        v = u + g
        grad = 1.0 - c / v + a * k_of(u)
        h = c / (v * v)
        pre = 1.0 / (h + a * 2.0 * q.mean())
        # conjugate gradients on (diag(h) + alpha K) s = -grad
        s = torch.zeros_like(u)
        res = -grad
        z = pre * res
        p = z.clone()
        rz = dot(res, z)
        first = rz.clone()
        for it in range(200):
            ap = h * p + a * k_of(p)
            t = rz / dot(p, ap).clamp(min=1e-300)
            s = s + t * p
            res = res - t * ap
            z = pre * res
            new = dot(res, z)
            if it % 10 == 9 and bool((new <= 1e-26 * first).all()):
                break
            p = z + (new / rz.clamp(min=1e-300)) * p
            rz = new
        # stay inside the barrier, and halve the step where the cost rises
        worst = (-s / v).amax(dim=(1, 2), keepdim=True).clamp(min=1e-300)
        step = torch.minimum(torch.ones_like(worst), 0.9 / worst)
        f0 = cost_of(u)
        for _ in range(20):
            worse = cost_of(u + step * s) > f0 + 1e-13 * f0.abs()
            if not bool(worse.any()):
                break
            step = torch.where(worse, 0.5 * step, step)
        u = u + step * s
        if bool((dot(s, s) <= 1e-22 * dot(u, u)).all()):
            break
    return u, cost_of(u).reshape(-1)


def _exact_frame(data, gamma, mask_fft, alpha, r=16):
    """Reference tiling of one frame: windows of side r at stride r - 2 on the
    frame with one replicated pixel around it, the last window clamped, later
    windows owning the overlaps."""
    h, w = data.shape
    s = r - 2

    def starts(n):
        k = 1 + -(-(n - s) // s)
        return [min(-1 + s * i, n + 1 - r) for i in range(k)]

    ys, xs = starts(h), starts(w)
    rows = (torch.tensor(ys, device=DEV)[:, None] + torch.arange(r, device=DEV)).clamp(0, h - 1)
    cols = (torch.tensor(xs, device=DEV)[:, None] + torch.arange(r, device=DEV)).clamp(0, w - 1)
    pick = lambda a: a.double()[rows[:, None, :, None], cols[None, :, None, :]].reshape(-1, r, r)
    d, g = pick(data), pick(gamma)
    us, costs = [], []
    for i in range(0, len(d), 20000):
        u, cost = _minimise(d[i:i + 20000], g[i:i + 20000], mask_fft, alpha)
        us.append(u)
        costs.append(cost)
    u = torch.cat(us).view(len(ys), len(xs), r, r)

    # each axis: the window that owns a pixel is the last one whose interior
    # holds it
    def owner(first, n):
        own = torch.zeros(n, dtype=torch.long, device=DEV)
        at = torch.zeros(n, dtype=torch.long, device=DEV)
        for k, b in enumerate(first):
            own[b + 1:b + r - 1] = k
            at[b + 1:b + r - 1] = torch.arange(1, r - 1, device=DEV)
        return own, at

    oy, ay = owner(ys, h)
    ox, ax = owner(xs, w)
    img = u[oy[:, None], ox[None, :], ay[:, None], ax[None, :]]
    return img, torch.cat(costs)


def _exact_net(x, target, params):
    """Output, loss and parameter gradient of the conv net in float64."""
    p = params.detach().double().requires_grad_(True)
    h = x.double()
    for i, (ws, bs, cin, cout) in enumerate(warmstart.layer_slices()):
        wt = p[ws].view(cout, cin, 9)
        # the 3 x 3 convolution as a product over unfolded pixels
        cols = torch.nn.functional.unfold(h, 3, padding=1).view(h.shape[0], cin * 9, 256)
        h = (torch.matmul(wt.reshape(cout, cin * 9), cols) + p[bs][None, :, None])
        h = h.view(x.shape[0], cout, 16, 16)
        if i < 3:
            h = torch.relu(h)
    y = h[:, 0]
    loss = torch.mean((y - target.double()) ** 2)
    loss.backward()
    return y.detach(), loss.detach(), p.grad


def exact(case, seed):
    path = case["path"]
    fft = lambda kind: masks.to_fft_order(_mask(kind))
    if path == "train":
        y, loss, grad = _exact_net(*_train_inputs(case, seed))
        return dict(y=y, loss=loss, grad=grad)
    if path == "tiles":
        data, gamma = _tiles(case, seed)
        u, cost = _minimise(data.double(), gamma.double(), fft("gauss"), case["alpha"])
        return dict(u=u, status=None, cost=cost)
    if path == "clib":
        data, gamma = _same_size(case, seed)
        mask = masks.to_fft_order(masks.otf_mask(r=case["window"]))
        return _exact_frame(data[0], gamma, mask, case["alpha"], case["window"])[0]
    if path == "stream":
        raw, offset, gain, var = _raw_series(case, seed)
        data = [(r.double() - offset) / gain for r in raw]
        return [_exact_frame(torch.where(d <= 0, torch.full_like(d, 1.0e-6), d),
                             var / gain ** 2, fft("otf"), case["alpha"])[0] for d in data]
    if path == "host":
        data, gamma = _same_size(case, seed)
        return [_exact_frame(d, gamma, fft("otf"), case["alpha"])[0] for d in data]
    if path == "device":
        data, gamma = _same_size(case, seed)
        got = [_exact_frame(d, gamma, fft(case["mask"]), case["alpha"]) for d in data]
    else:
        data, gamma, _, alphas = _uneven(case, seed)
        got = [_exact_frame(d, g, fft("otf"), a) for d, g, a in zip(data, gamma, alphas)]
    return dict(out=[x[0] for x in got], status=None, cost=torch.cat([x[1] for x in got]))
