"""The work a user has this library do on one GPU, as measurable cases.

Kinds of case, and what each stands for:

* corr      the ``Correlation`` custom op on one level of a feature pyramid
            (float32, bfloat16, float16, or float32 features quantised to
            FP8 E4M3 and correlated);
* warp      the ``Warp`` custom op on one level;
* stab      one stabilized frame with flows given (``do_one_step``), reference
            operation order or FMA form;
* flownet   the flow network of one frame: the new frame's features and the
            forward and backward flows;
* upsample  the learned flow upsampler for one flow;
* train     one loss and gradient of the upsampler's training;
* pipeline  a whole frame: flows computed, upsampled, frame stabilized.

Sizes are those of the feature pyramid of a 1920x1088 pair, of the 640x360
and 1920x1080 synthetic workloads and of the serving mix (640x360 to
3840x2160), and odd ones between them.
"""
import functools
import importlib
import math

import numpy as np
import torch
import torch.nn.functional as F

vsc = importlib.import_module("video-stream-consistency_amd")

# one pyramid of a 1920x1088 pair: (channels, height, width)
_PYRAMID = [(32, 272, 480), (64, 136, 240), (96, 68, 120), (128, 34, 60), (196, 17, 30)]
_TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_HEAD_SCALE = 0.05  # untrained flow heads brought to the magnitude of real motion


def _corr(C, H, W, dtype, N=1, legacy=0):
    return {"kind": "corr", "N": N, "C": C, "H": H, "W": W, "dtype": dtype, "legacy": legacy}


def _stab(W, H, fma, levels=2, iters=150, gamma=2.0, down=1):
    return {"kind": "stab", "W": W, "H": H, "fma": fma, "levels": levels, "iters": iters, "gamma": gamma, "down": down}


def listed():
    return [
        # the coarsest level of a pyramid: the smallest call, bound by its launch and its latency
        {"name": "corr_f32_30x17", **_corr(196, 17, 30, "f32")},
        # the finest level a decoder correlates at, in the op's own type
        {"name": "corr_f32_480x272", **_corr(32, 272, 480, "f32")},
        # a middle level of an odd-sized stream's pyramid in 16 bits (rows that are not aligned)
        {"name": "corr_bf16_213x119", **_corr(64, 119, 213, "bf16")},
        # warping the second frame's features towards the first
        {"name": "warp_f32_480x272", "kind": "warp", "N": 1, "C": 32, "H": 272, "W": 480},
        # a small stream, flows from files, the default (reference order) solver
        {"name": "stab_exact_640x360", **_stab(640, 360, False)},
        # the ordinary frame: Full HD, flows given, the pipeline's solver
        {"name": "stab_fma_1920x1080", **_stab(1920, 1080, True)},
        # the largest stream of the serving mix
        {"name": "stab_fma_3840x2160", **_stab(3840, 2160, True)},
        # the flow network of a Full-HD frame as it is recommended to run: half resolution, 16-bit
        {"name": "flownet_bf16_1920x1080", "kind": "flownet", "W": 1920, "H": 1080, "down": 2, "dtype": "bf16"},
        # the flow network of a small stream at full resolution in 32 bits
        {"name": "flownet_f32_640x360", "kind": "flownet", "W": 640, "H": 360, "down": 1, "dtype": "f32"},
        # bringing a half-resolution flow to a Full-HD frame
        {"name": "upsample_1920x1080", "kind": "upsample", "W": 1920, "H": 1080, "down": 2},
        # training the upsampler on a batch of crops: forward, backward, gradient
        {"name": "train_8x128x128", "kind": "train", "B": 8, "W": 128, "H": 128},
        # one Full-HD frame end to end in the form that is recommended
        {"name": "pipeline_1920x1080", "kind": "pipeline", "W": 1920, "H": 1080, "form": "chosen"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["corr", "corr", "warp", "stab", "stab", "stab", "flownet", "upsample", "train", "pipeline"])
    if kind in ("corr", "warp"):
        H, W = _log(rng, 17, 272), _log(rng, 30, 480)
        C = rng.choice([16, 32, 64, 96, 128, 196, rng.randrange(8, 200)])
        C = max(4, min(C, 32 * 272 * 480 // (H * W)))
        N = 2 if 2 * H * W * C <= 32 * 272 * 480 and rng.random() < 0.3 else 1
        if kind == "warp":
            return {"kind": "warp", "N": N, "C": C, "H": H, "W": W}
        dtype = rng.choice(["f32", "f32", "bf16", "f16", "fp8"])
        return _corr(C, H, W, dtype, N, 1 if rng.random() < 0.15 else 0)
    if kind == "stab":
        fma = rng.random() < 0.6
        W = _log(rng, 160, 3840 if fma else 1920)
        H = max(64, min(2160 if fma else 1080, int(W * rng.choice([9 / 16, 9 / 16, 3 / 4, 0.5]))))
        H += rng.choice([0, 0, 1, -1])
        return _stab(W, H, fma, rng.choice([1, 2, 2, 2, 3]), rng.choice([150, 150, 100, rng.randrange(20, 150)]),
                     rng.choice([2.0, 2.0, 0.5, 8.0]), rng.choice([1, 1, 2]))
    if kind == "flownet":
        dtype = rng.choice(["bf16", "f32"])
        down = rng.choice([1, 2])
        W = _log(rng, 256, 960 * down)
        H = max(144, int(W * rng.choice([9 / 16, 3 / 4] if W < 800 * down else [9 / 16])))
        return {"kind": "flownet", "W": W, "H": H, "down": down, "dtype": dtype}
    if kind == "upsample":
        W = _log(rng, 160, 1920)
        return {"kind": "upsample", "W": W, "H": max(90, int(W * rng.choice([9 / 16, 0.5]))), "down": rng.choice([2, 2, 4])}
    if kind == "train":
        return {"kind": "train", "B": rng.choice([1, 2, 4, 8]), "W": rng.randrange(48, 129), "H": rng.randrange(48, 129)}
    form = rng.choice(["chosen", "chosen", "plain"])
    W = _log(rng, 320, 1920 if form == "chosen" else 960) // 2 * 2
    return {"kind": "pipeline", "W": W, "H": max(180, int(W * 9 / 16)) // 2 * 2, "form": form}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _smooth(g, ch, H, W, cell):
    """A smooth random field: bicubic interpolation of a coarse normal grid."""
    low = torch.randn((1, ch, H // cell + 4, W // cell + 4), generator=g, device="cuda")
    return F.interpolate(low, size=(H, W), mode="bicubic", align_corners=True)[0]


def _video(seed, n, H, W):
    """n frames of textured content in smooth motion and their flickering
    processed versions (RGBA8), and the flows between neighbours (HWC)."""
    g = _gen(seed)
    tex = 0.5 + 0.16 * _smooth(g, 3, H, W, max(4, W // 24)) + 0.10 * _smooth(g, 3, H, W, 9)
    v = (torch.rand(2, generator=g, device="cuda") * 2 - 1) * 8.0 * (W / 1920.0)
    d = v[:, None, None] + 0.7 * _smooth(g, 2, H, W, max(8, W // 10))
    ys, xs = torch.meshgrid(torch.arange(H, device="cuda"), torch.arange(W, device="cuda"), indexing="ij")
    orig, proc = [], []
    for t in range(n):
        gx, gy = (xs - t * d[0]) * (2.0 / (W - 1)) - 1, (ys - t * d[1]) * (2.0 / (H - 1)) - 1
        im = F.grid_sample(tex[None], torch.stack([gx, gy], -1)[None], mode="bilinear", padding_mode="reflection", align_corners=True)[0]
        gain = 0.8 + 0.4 * torch.rand(3, 1, 1, generator=g, device="cuda")
        off = (torch.rand(3, 1, 1, generator=g, device="cuda") - 0.5) * (40 / 255)
        pr = im * gain + off + (4 / 255) * torch.randn(im.shape, generator=g, device="cuda")
        for x, to in ((im, orig), (pr, proc)):
            b = torch.full((H, W, 4), 255, dtype=torch.uint8, device="cuda")
            b[..., :3] = (x.clamp(0, 1) * 255).round().to(torch.uint8).permute(1, 2, 0)
            to.append(b)
    fwd = d.permute(1, 2, 0).contiguous()
    return orig, proc, fwd, (-fwd).contiguous()


def _features(case, seed):
    g = _gen(seed)
    shape = (case["N"], case["C"], case["H"], case["W"])
    return [F.leaky_relu(torch.randn(shape, generator=g, device="cuda"), 0.1) for _ in range(2)], g


def _op_flow(case, g):
    N, H, W = case["N"], case["H"], case["W"]
    return torch.stack([2.0 * _smooth(g, 2, H, W, 16) for _ in range(N)]) + torch.rand((N, 2, H, W), generator=g, device="cuda") - 0.5


def _low(flow, down, ch=2):
    """A flow at the network's resolution, its vectors in that resolution's pixels."""
    H, W = flow.shape[:2]
    t = F.interpolate(flow.permute(2, 0, 1)[None], size=(int(round(H / down)), int(round(W / down))), mode="bilinear", align_corners=False)
    return (t[0].permute(1, 2, 0) / down).contiguous()


_FEAT = [3, 16, 32, 64, 96, 128, 196]
_DEC = [128, 128, 96, 64, 32, 2]
_REF = [128, 128, 128, 96, 64, 32, 2]
_DIL = [1, 2, 4, 8, 16, 1, 1]


def _layers():
    """(weight shape, whether a flow head) in the order vsc_flownet_set_params takes."""
    out = []
    for k in range(1, 7):
        out += [((_FEAT[k], _FEAT[k - 1] if j == 0 else _FEAT[k], 3, 3), False) for j in range(3)]
    out += [((2, 2, 4, 4), False)] * 3
    for lvl in (6, 5, 4, 3):
        cin = [83 + _FEAT[lvl], 128, 256, 224, 160, 96]
        out += [((_DEC[j], cin[j], 3, 3), j == 5) for j in range(6)]
    out += [((_REF[j], 34 if j == 0 else _REF[j - 1], 3, 3), j == 6) for j in range(7)]
    return out


@functools.lru_cache(maxsize=1)
def _weights():
    """The network's weights, as a program loads them from its file: Kaiming
    normal for LeakyReLU(0.1), small biases, scaled-down flow heads."""
    rng = np.random.default_rng(11)
    parts = []
    for (co, ci, kh, kw), head in _layers():
        s = math.sqrt(2.0 / 1.01 / (ci * kh * kw)) * (_HEAD_SCALE if head else 1.0)
        parts.append(rng.standard_normal(co * ci * kh * kw, dtype=np.float32) * np.float32(s))
        parts.append(rng.standard_normal(co, dtype=np.float32) * np.float32(0.01 * (_HEAD_SCALE if head else 1.0)))
    return np.concatenate(parts)


def _params(case):
    return vsc.HyperParams(gamma=case["gamma"], pyramidLevels=case["levels"], numIter=case["iters"])


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": case}
    if kind == "corr":
        f, _ = _features(case, seed)
        s["f"] = f if case["dtype"] == "fp8" else [x.to(_TORCH[case["dtype"]]) for x in f]
    elif kind == "warp":
        f, g = _features(case, seed)
        s["f"], s["flow"] = f[0], _op_flow(case, g)
    elif kind == "stab":
        W, H = case["W"], case["H"]
        o, p, fwd, bwd = _video(seed, 3, H, W)
        if case["down"] > 1:
            fwd, bwd = _low(fwd, case["down"]), _low(bwd, case["down"])
        st = vsc.VideoStabilizer(W, H, fwd.shape[1], fwd.shape[0], mode=vsc.VSC_FRAME_FMA if case["fma"] else vsc.VSC_FRAME_FUSED)
        st.set_last_rgba(p[2])
        s.update(st=st, o=o, p=p, fwd=fwd, bwd=bwd, prm=_params(case), rgba=torch.empty_like(o[0]),
                 frame=torch.empty((H, W, 3), device="cuda"))
    elif kind == "flownet":
        s["o"] = _video(seed, 4, case["H"], case["W"])[0]
        net = vsc.FlowNet(case["W"], case["H"], case["down"], case["dtype"], slots=3)
        net.set_params(_weights())
        for k in range(2):
            net.extract(s["o"][k], k)
        s.update(net=net, t=2)
    elif kind == "upsample":
        o, _, fwd, _ = _video(seed, 1, case["H"], case["W"])
        s.update(up=vsc.Upsampler(params=vsc.load_upsampler_weights()), lo=_low(fwd, case["down"]), rgba=o[0])
    elif kind == "train":
        s.update(zip(("lo", "rgba", "gt"), _train_batch(case, seed)))
        s["up"] = vsc.Upsampler(params=vsc.load_upsampler_weights())
    else:
        s["o"], s["p"], _, _ = _video(seed, 6, case["H"], case["W"])
        s["pipe"] = _pipeline(case)
        s["pipe"].set_last_rgba(s["p"][2])
        s.update(t=1, rgba=torch.empty_like(s["o"][0]), frame=torch.empty((case["H"], case["W"], 3), device="cuda"))
    return s


def _train_batch(case, seed):
    lo, rgba, gt = [], [], []
    for b in range(case["B"]):
        o, _, fwd, _ = _video(seed * 31 + b, 1, case["H"], case["W"])
        lo.append(_low(fwd, 2))
        rgba.append(o[0])
        gt.append(fwd)
    return torch.stack(lo), torch.stack(rgba), torch.stack(gt)


def _pipeline(case):
    import ctypes
    pipe = vsc.Pipeline(case["W"], case["H"], form=case["form"])
    net = ctypes.c_void_p()
    vsc.check(vsc.lib().vsc_pipeline_flownet(pipe.h, ctypes.byref(net)))
    w = _weights()
    vsc.check(vsc.lib().vsc_flownet_set_params(net, w.ctypes.data, w.size))
    return pipe


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "corr":
        if case["dtype"] == "fp8":
            q1, q2, sc = vsc.quantize_fp8_pair(s["f"][0], s["f"][1])
            return {"q1": q1, "q2": q2, "scale": sc, "out": vsc.correlation_fp8(q1, q2, sc, 4, case["legacy"])}
        return {"out": vsc.correlation(s["f"][0], s["f"][1], 4, case["legacy"])}
    if kind == "warp":
        return {"out": vsc.warp(s["f"], s["flow"])}
    if kind == "stab":
        s["st"].do_one_step(s["o"], s["p"], s["fwd"], s["bwd"], out_rgba=s["rgba"], out_float=s["frame"], params=s["prm"])
        return {"rgba": s["rgba"], "frame": s["frame"]}
    if kind == "flownet":
        # slots rotate: the new frame's features, then the flows of the window around the frame before it
        t = s["t"]
        s["t"] = t + 1
        s["net"].extract(s["o"][t % 4], t % 3)
        fwd, bwd = s["net"].flow([((t - 1) % 3, t % 3), ((t - 1) % 3, (t - 2) % 3)])
        return {"fwd": fwd, "bwd": bwd}
    if kind == "upsample":
        return {"flow": s["up"].run(s["lo"], s["rgba"], scale=float(case["down"]))}
    if kind == "train":
        loss, grad = s["up"].loss_grad(s["lo"], s["rgba"], s["gt"])
        return {"loss": loss, "grad": grad}
    t = s["t"]
    s["t"] = t + 1
    o, p = s["o"], s["p"]
    w = (o[(t - 1) % 6], o[t % 6], o[(t + 1) % 6], p[(t - 1) % 6], p[t % 6], p[(t + 1) % 6])
    s["pipe"].frame(w, t, out_rgba=s["rgba"], out_float=s["frame"])
    return {"rgba": s["rgba"], "frame": s["frame"]}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _stab_work(W, H, levels, iters, flow_bytes):
    px = W * H
    # 6 RGBA8 frames, the flows, the previous frame in; RGBA8, the float frame and the new previous frame out
    by = px * (24 + 12 + 4 + 12 + 12) + flow_bytes
    # front pass about 400 operations a pixel; a solver sweep is 3 additions, an addition and 3 fused operations a value
    return {"bytes": by, "flops": 400 * px + sum(10 * 3 * (px >> 2 * j) * (iters // (j + 1)) for j in range(levels))}


def _net_work(W, H, down, size, pairs=2):
    w, h = int(round(W / down)), int(round(H / down))
    wp, hp = (w + 63) // 64 * 64, (h + 63) // 64 * 64
    fl, params = 0, 0
    shapes = [s for s, _ in _layers()]
    for k in range(1, 7):
        fl += sum(2 * math.prod(s) * (wp >> k) * (hp >> k) for s in shapes[3 * k - 3:3 * k])
    for i, lvl in enumerate((6, 5, 4, 3)):
        px = (wp >> lvl) * (hp >> lvl)
        fl += pairs * px * (sum(2 * math.prod(s) for s in shapes[21 + 6 * i:27 + 6 * i]) + 2 * 81 * _FEAT[lvl])
    fl += pairs * (wp >> 3) * (hp >> 3) * sum(2 * math.prod(s) for s in shapes[45:])
    params = sum(math.prod(s) for s in shapes) * size
    # the new frame and the weights in, two cached frames' features in, the new frame's out, the flows out
    feats = sum(_FEAT[l] * (wp >> l) * (hp >> l) for l in (3, 4, 5, 6)) * size
    return {"bytes": W * H * 4 + params + 3 * feats + pairs * w * h * 8, "flops": fl}


def work(case):
    kind = case["kind"]
    if kind in ("corr", "warp"):
        N, C, px = case["N"], case["C"], case["H"] * case["W"]
        if kind == "warp":
            return {"bytes": N * px * (8 * C + 8), "flops": N * px * (8 * C + 20)}
        size = {"f32": 4, "bf16": 2, "f16": 2, "fp8": 4}[case["dtype"]]
        quant = 2 * C if case["dtype"] == "fp8" else 0
        return {"bytes": N * px * (2 * C * size + quant + 81 * 4), "flops": N * px * 2 * 81 * C}
    W, H = case["W"], case["H"]
    if kind == "stab":
        return _stab_work(W, H, case["levels"], case["iters"], 16 * W * H // case["down"] ** 2)
    if kind == "flownet":
        return _net_work(W, H, case["down"], 2 if case["dtype"] == "bf16" else 4)
    ups = 2 * (27 * 16 + 144 * 16 + 144 * 2) * W * H
    if kind == "upsample":
        return {"bytes": W * H * (8 / case["down"] ** 2 + 4 + 8), "flops": ups}
    if kind == "train":
        return {"bytes": case["B"] * W * H * (2 + 4 + 8), "flops": 3 * ups * case["B"]}
    chosen = case["form"] == "chosen"
    n = _net_work(W, H, 2 if chosen else 1, 2 if chosen else 4)
    b = _stab_work(W, H, 2, 150, 0)
    return {"bytes": n["bytes"] + b["bytes"], "flops": n["flops"] + b["flops"] + (2 * ups if chosen else 0)}


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _shift_corr(a, b, legacy):
    N, C, H, W = a.shape
    p = F.pad(b, (4, 4, 4, 4))
    out = torch.stack([(a * p[:, :, dy:dy + H, dx:dx + W]).sum(1) for dy in range(9) for dx in range(9)], 1)
    return out / C if legacy else out.view(N, 9, 9, H, W)


def _op_warp(x, flow):
    """x NCHW and flow N2HW in 64 bits: bilinear, zero outside, zero where the mass inside is below 0.999."""
    N, C, H, W = x.shape
    ys, xs = torch.meshgrid(torch.arange(H, device=x.device, dtype=x.dtype), torch.arange(W, device=x.device, dtype=x.dtype), indexing="ij")
    px, py = xs + flow[:, 0], ys + flow[:, 1]
    x0, y0 = px.floor(), py.floor()
    fx, fy = px - x0, py - y0
    out, mass = 0, 0
    for dx, dy in ((0, 0), (1, 0), (0, 1), (1, 1)):
        ix, iy = x0 + dx, y0 + dy
        wt = (fx if dx else 1 - fx) * (fy if dy else 1 - fy)
        wt = torch.where((ix >= 0) & (ix <= W - 1) & (iy >= 0) & (iy <= H - 1), wt, torch.zeros_like(wt))
        at = (iy.clamp(0, H - 1) * W + ix.clamp(0, W - 1)).long().view(N, 1, -1).expand(-1, C, -1)
        out = out + wt[:, None] * torch.gather(x.reshape(N, C, -1), 2, at).view_as(x)
        mass = mass + wt
    return out * (mass > 0.999)[:, None]


def _resample(x, H, W):
    """CHW bilinear resampling with source position o * in / out."""
    def taps(n, m):
        o = torch.arange(n, device=x.device, dtype=x.dtype) * m / n
        i = o.floor()
        return i.long(), (i.long() + 1).clamp(max=m - 1), o - i
    x0, x1, fx = taps(W, x.shape[2])
    y0, y1, fy = taps(H, x.shape[1])
    rows = x[:, y0] * (1 - fy)[:, None] + x[:, y1] * fy[:, None]
    return rows[:, :, x0] * (1 - fx) + rows[:, :, x1] * fx


def _frame_warp(x, flow):
    """CHW sampled at the position clamped to [0, W-3] x [0, H-3]."""
    C, H, W = x.shape
    ys, xs = torch.meshgrid(torch.arange(H, device=x.device, dtype=x.dtype), torch.arange(W, device=x.device, dtype=x.dtype), indexing="ij")
    px, py = (xs + flow[..., 0]).clamp(max=W - 3).clamp(min=0), (ys + flow[..., 1]).clamp(max=H - 3).clamp(min=0)
    x0, y0 = px.floor(), py.floor()
    fx, fy = px - x0, py - y0
    at = (y0 * W + x0).long().view(-1)
    v = x.reshape(C, -1)
    t1 = v[:, at].view_as(x) * (1 - fx) + v[:, at + 1].view_as(x) * fx
    t2 = v[:, at + W].view_as(x) * (1 - fx) + v[:, at + W + 1].view_as(x) * fx
    return t1 * (1 - fy) + t2 * fy


def _neighbours(x):
    """Sum over the solver's neighbours of each pixel: the right and lower ones only up to the last but one."""
    s = torch.zeros_like(x)
    s[..., :, :-2] += x[..., :, 1:-1]
    s[..., :, 1:] += x[..., :, :-1]
    s[..., :-2, :] += x[..., 1:-1, :]
    s[..., 1:, :] += x[..., :-1, :]
    return s


def _exact_stab(o, p, fwd, bwd, last, gamma=2.0, levels=2, iters=150, alpha=6800.0, beta=6800.0, step=0.15, mom=0.15):
    o, p = [[x[..., :3].permute(2, 0, 1).double() / 255 for x in v] for v in (o, p)]
    pi, pp, ls = (_frame_warp(x, bwd) for x in (o[0], p[0], last))
    ni, np_ = (_frame_warp(x, fwd) for x in (o[2], p[2]))
    wp = torch.exp(-alpha * (o[1] - pi) ** 2).clamp(max=0.45)
    wn = torch.exp(-alpha * (o[1] - ni) ** 2).clamp(max=0.3)
    wp, wn = (torch.where(w < 0.001, torch.zeros_like(w), w) for w in (wp, wn))
    ad = wp * pi + wn * ni + (1 - wp - wn) * o[1]
    A = wp * ls + (1 - wp) * (wp * pp + wn * np_ + (1 - wp - wn) * p[1])
    Wt = gamma * torch.exp(-beta * (o[1] - ad) ** 2)
    Wt = torch.where(Wt < 0.001, torch.zeros_like(Wt), Wt)
    lev = [(p[1], A, Wt)]
    for _ in range(1, levels):
        H, W = lev[-1][0].shape[1:]
        lev.append(tuple(_resample(x, H // 2, W // 2) for x in lev[-1]))
    O = lev[-1][0]
    for j in range(levels - 1, -1, -1):
        P, A, Wt = lev[j]
        if j < levels - 1:
            O = _resample(O, *P.shape[1:])
        cnt = _neighbours(torch.ones_like(P))
        const = Wt * A - (_neighbours(P) - cnt * P)
        q, U = cnt + Wt, torch.zeros_like(P)
        for _ in range(iters // (j + 1)):
            G = step * (_neighbours(O) - q * O + const)
            O, U = O + G + mom * U, G
    return O.permute(1, 2, 0).contiguous()


def _conv(x, w, b, stride=1, dil=1):
    """3x3 convolution in 64 bits as a matrix product, some rows of the output at a time."""
    x = F.pad(x, (dil, dil, dil, dil))
    N, C, H, W = x.shape
    ho, wo = (H - 2 * dil - 1) // stride + 1, (W - 2 * dil - 1) // stride + 1
    out = x.new_empty((N, w.shape[0], ho, wo))
    rows = max(1, (1 << 25) // (9 * C * wo))
    m = w.reshape(w.shape[0], -1)
    for n in range(N):
        for r in range(0, ho, rows):
            k = min(rows, ho - r)
            cols = torch.stack([x[n, :, r * stride + dy * dil:(r + k - 1) * stride + dy * dil + 1:stride,
                                  dx * dil:(wo - 1) * stride + dx * dil + 1:stride] for dy in range(3) for dx in range(3)], 1)
            out[n, :, r:r + k] = (m @ cols.reshape(9 * C, k * wo)).view(-1, k, wo) + b[:, None, None]
    return out


def _exact_flows(frames, pairs, down):
    """The flows (HWC) of the (first, second) pairs of RGBA8 frames."""
    flat, P, at = torch.from_numpy(_weights()).cuda().double(), [], 0
    for shape, _ in _layers():
        n = math.prod(shape)
        nb = shape[0]
        P.append((flat[at:at + n].view(shape), flat[at + n:at + n + nb]))
        at += n + nb
    act = lambda v: F.leaky_relu(v, 0.1)  # noqa: E731
    H, W = frames[0].shape[:2]
    h, w = int(round(H / down)), int(round(W / down))
    hp, wp = (h + 63) // 64 * 64, (w + 63) // 64 * 64
    feats = []
    for im in frames:
        if down > 1:
            ys, xs = (np.minimum(n - 1, ((np.arange(m, dtype=np.float32) + np.float32(0.5)) * np.float32(np.float32(n) / np.float32(m))).astype(np.int64))
                      for n, m in ((H, h), (W, w)))
            im = im[torch.from_numpy(ys).cuda()][:, torch.from_numpy(xs).cuda()]
        x = F.interpolate(im[..., :3].permute(2, 0, 1)[None].double() / 255, size=(hp, wp), mode="bilinear", align_corners=False)
        f = [None]
        for k in range(6):
            for j in range(3):
                x = act(_conv(x, *P[3 * k + j], stride=2 if j == 0 else 1))
            f.append(x)
        feats.append(f)
    out = []
    for a, b in pairs:
        fl = x5 = None
        for i, lvl in enumerate((6, 5, 4, 3)):
            f1, f2 = feats[a][lvl], feats[b][lvl]
            D = P[21 + 6 * i:27 + 6 * i]
            if fl is None:
                up = torch.zeros((1, 2) + f1.shape[2:], dtype=f1.dtype, device=f1.device)
            else:
                wt, bias = P[18 + i - 1]  # transposed convolution, 4x4, stride 2, padding 1
                z = torch.zeros((1, 2, 2 * fl.shape[2] + 2, 2 * fl.shape[3] + 2), dtype=fl.dtype, device=fl.device)
                for ky in range(4):
                    for kx in range(4):
                        z[0, :, ky:ky + 2 * fl.shape[2]:2, kx:kx + 2 * fl.shape[3]:2] += torch.tensordot(wt[:, :, ky, kx], fl[0], ([0], [0]))
                up = z[:, :, 1:-1, 1:-1] + bias[:, None, None]
                f2 = _op_warp(f2, up * {5: 0.625, 4: 1.25, 3: 2.5}[lvl])
            x1 = act(_conv(torch.cat([act(_shift_corr(f1, f2, 0).flatten(1, 2)), f1, up], 1), *D[0]))
            x2 = act(_conv(x1, *D[1]))
            x3 = act(_conv(torch.cat([x1, x2], 1), *D[2]))
            x4 = act(_conv(torch.cat([x2, x3], 1), *D[3]))
            x5 = act(_conv(torch.cat([x3, x4], 1), *D[4]))
            fl = _conv(torch.cat([x4, x5], 1), *D[5])
        x = torch.cat([x5, fl], 1)
        for j in range(7):
            x = _conv(x, *P[45 + j], dil=_DIL[j])
            x = act(x) if j < 6 else x
        up = F.interpolate((fl + x) * 20.0, scale_factor=8, mode="bilinear", align_corners=True)
        y = F.interpolate(up, size=(h, w), mode="bilinear", align_corners=False)[0]
        out.append((y * torch.tensor([h / hp, w / wp], dtype=y.dtype, device=y.device)[:, None, None]).permute(1, 2, 0))
    return out


def _ups_params(grad=False):
    flat = torch.from_numpy(vsc.load_upsampler_weights()).cuda().double()
    out, at = [], 0
    for shape in ((16, 3, 3, 3), (16,), (16, 16, 3, 3), (16,), (2, 16, 3, 3), (2,)):
        out.append(flat[at:at + math.prod(shape)].view(shape).clone().requires_grad_(grad))
        at += math.prod(shape)
    return out


def _exact_upsample(P, lo, rgba, scale):
    """HWC flow of one frame (differentiable in P)."""
    H, W = rgba.shape[:2]
    base = scale * _resample(lo.double().permute(2, 0, 1), H, W)
    luma = (rgba[..., :3].double() @ torch.tensor([0.299, 0.587, 0.114], dtype=torch.float64, device="cuda")) / 255
    x = torch.cat([base, luma[None]])
    for i in range(3):
        p = F.pad(x, (1, 1, 1, 1))
        cols = torch.stack([p[:, dy:dy + H, dx:dx + W] for dy in range(3) for dx in range(3)], 1).reshape(-1, H * W)
        x = (P[2 * i].reshape(P[2 * i].shape[0], -1) @ cols).view(-1, H, W) + P[2 * i + 1][:, None, None]
        x = torch.relu(x) if i < 2 else x
    return (base + x).permute(1, 2, 0)


def _inconsistent(f, b):
    """Share of the pixels whose forward and backward flows do not agree."""
    H, W = f.shape[:2]
    ys, xs = torch.meshgrid(torch.arange(H, device=f.device, dtype=f.dtype), torch.arange(W, device=f.device, dtype=f.dtype), indexing="ij")
    px, py = xs + f[..., 0], ys + f[..., 1]
    grid = torch.stack([px * 2 / (W - 1) - 1, py * 2 / (H - 1) - 1], -1)[None]
    v = F.grid_sample(b.permute(2, 0, 1)[None], grid, mode="bilinear", padding_mode="border", align_corners=True)[0].permute(1, 2, 0)
    off = ((f + v) ** 2).sum(-1) >= 0.01 * ((f ** 2).sum(-1) + (v ** 2).sum(-1)) + 0.5
    return float((off | (px < 0) | (px > W - 1) | (py < 0) | (py > H - 1)).double().mean())


def exact(case, seed):
    kind = case["kind"]
    if kind == "corr":
        (a, b), _ = _features(case, seed)
        if case["dtype"] == "fp8":  # against the features before they are quantised
            return {"q1": None, "q2": None, "scale": None, "out": _shift_corr(a.double(), b.double(), case["legacy"])}
        t = _TORCH[case["dtype"]]
        return {"out": _shift_corr(a.to(t).double(), b.to(t).double(), case["legacy"])}
    if kind == "warp":
        f, g = _features(case, seed)
        return {"out": _op_warp(f[0].double(), _op_flow(case, g).double())}
    W, H = case["W"], case["H"]
    if kind == "stab":
        o, p, fwd, bwd = _video(seed, 3, H, W)
        fl = [fwd.double(), bwd.double()]
        if case["down"] > 1:
            fl = [_resample(_low(x, case["down"]).double().permute(2, 0, 1), H, W).permute(1, 2, 0) for x in (fwd, bwd)]
        last = p[2][..., :3].permute(2, 0, 1).double() / 255
        return {"rgba": None, "frame": _exact_stab(o, p, fl[0], fl[1], last, case["gamma"], case["levels"], case["iters"])}
    if kind == "flownet":
        o = _video(seed, 4, H, W)[0]
        fwd, bwd = _exact_flows(o[:3], [(1, 2), (1, 0)], case["down"])
        return {"fwd": fwd, "bwd": bwd}
    if kind == "upsample":
        o, _, fwd, _ = _video(seed, 1, H, W)
        return {"flow": _exact_upsample(_ups_params(), _low(fwd, case["down"]), o[0], float(case["down"]))}
    if kind == "train":
        lo, rgba, gt = _train_batch(case, seed)
        P = _ups_params(grad=True)
        out = torch.stack([_exact_upsample(P, lo[b], rgba[b], 2.0) for b in range(case["B"])])
        loss = torch.sqrt(((out - gt.double()) ** 2).sum(-1) + 1e-6).mean()
        grad = torch.autograd.grad(loss, P)
        return {"loss": loss.detach().reshape(()), "grad": torch.cat([x.reshape(-1) for x in grad])}
    o, p, _, _ = _video(seed, 6, H, W)
    chosen = case["form"] == "chosen"
    fl = _exact_flows(o[:3], [(1, 2), (1, 0)], 2 if chosen else 1)
    if chosen:
        if _inconsistent(*fl) <= 0.25:
            fl = [_exact_upsample(_ups_params(), x, o[1], 2.0) for x in fl]
        else:
            fl = [2.0 * _resample(x.permute(2, 0, 1), H, W).permute(1, 2, 0) for x in fl]
    last = p[2][..., :3].permute(2, 0, 1).double() / 255
    return {"rgba": None, "frame": _exact_stab(o[:3], p[:3], fl[0], fl[1], last)}
