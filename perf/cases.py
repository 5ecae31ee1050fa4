"""The work that users of the filter library have it do, as measurable cases.

A case names an entry point (``op``) and the sizes of one call.  ``listed()``
gives a fixed set, ``draw(rng)`` one more case of the same ranges,
``prepare`` the device state a program holds before the call, ``run`` the call
itself, ``work`` the bytes and operations the call cannot do without, and
``exact`` the 64-bit values of outputs that are computed real numbers.

Images are the synthetic content of the test workloads (``workloads.py``): a
horizontal gradient 0..200, rectangles and discs of random grey, Gaussian
noise; they are made on the device from the seed.  Radii, sigmas, ROI rules
and stage parameters are the ones the workloads, the measurement tool and the
tests use; odd sizes are in every range.
"""
import math

import numpy as np
import torch

import opencuda_amd as oc
from opencuda_amd import surrogate as sg

# The network's per-pixel work: 6 layers of 3x3, 32 channels (forward).
NET_FLOP = 2 * (18 * 32 + 4 * 288 * 32 + 288)
NET_PARAMS = 37889
CROP_MARGIN = 6          # crop border the training loss leaves out


def listed():
    return [
        # A thumbnail-sized inspection image, small window: launch latency and
        # a device that is not filled.
        {"name": "filter_512_r3", "op": "filter", "w": 512, "h": 512, "r": 3, "mode": "ref",
         "ss": 3.0, "sr": 30.0, "noise": 10.0},
        # One large ROI of a larger camera frame at the usual window size.
        {"name": "filter_roi3800x3600_r7", "op": "filter", "w": 3800, "h": 3600, "r": 7,
         "mode": "ref", "ss": 5.0, "sr": 25.0, "noise": 10.0, "pad_x": 296, "pad_y": 496},
        # The headline: a 31x31 window over a 67 Mpx image.
        {"name": "filter_8192_r15", "op": "filter", "w": 8192, "h": 8192, "r": 15, "mode": "ref",
         "ss": 10.0, "sr": 30.0, "noise": 12.0},
        # Own-window filtering at a radius without a kernel of its own, odd size.
        {"name": "filter_2047x1533_r11_std", "op": "filter", "w": 2047, "h": 1533, "r": 11,
         "mode": "std", "ss": 7.3, "sr": 25.0, "noise": 10.0},
        # The large end of the radii the class accepts (weight table beyond LDS).
        {"name": "filter_1500x1100_r18", "op": "filter", "w": 1500, "h": 1100, "r": 18,
         "mode": "ref", "ss": 12.0, "sr": 30.0, "noise": 10.0},
        # Many uneven images with ROIs and mixed radii in one planned launch.
        {"name": "batch_48", "op": "batch", "images": 48, "lo": 256, "hi": 2048, "mode": "ref"},
        # The class's in-place entry point with its repeat count.
        {"name": "inplace_1279x1024_r5_x3", "op": "inplace", "w": 1279, "h": 1024, "r": 5,
         "mode": "ref", "ss": 3.3, "sr": 20.0, "noise": 10.0, "repeat": 3},
        # The stage before the filter in the region detector, on a raw frame.
        {"name": "cluster_2048x1536", "op": "cluster", "w": 2048, "h": 1536, "range": 8,
         "count": 5, "gap": 10, "diffe": 10, "noise": 10.0},
        # The stage after it, on filtered (quiet) content.
        {"name": "regions_4096", "op": "regions", "w": 4096, "h": 4096, "noise": 2.0},
        # The detector's three stages on a mid-size frame, back to back.
        {"name": "chain_1021x767", "op": "chain", "w": 1021, "h": 767, "noise": 10.0},
        # Learned filter with the sampled check and the exact fallback.
        {"name": "surrogate_4096_r15", "op": "surrogate", "w": 4096, "h": 4096, "r": 15,
         "ss": 10.0, "sr": 30.0, "noise": 12.0},
        # One forward and backward pass of a training batch, early in training.
        {"name": "train_64x256", "op": "train", "n": 64, "h": 256, "w": 256},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["filter", "filter", "filter", "batch", "inplace", "cluster", "regions",
                     "chain", "surrogate", "train"])
    noise = round(rng.uniform(6.0, 14.0), 2)
    if op == "filter":
        mode = rng.choice(["ref", "std"])
        r = rng.randint(1, 19)
        return {"op": op, "w": _size(rng, 64, 4096), "h": _size(rng, 64, 4096), "r": r,
                "mode": mode, "ss": round(max(0.7, r / 1.5), 3),
                "sr": round(rng.uniform(10.0, 50.0), 3), "noise": noise,
                "pad_x": rng.randint(0, 64), "pad_y": rng.randint(0, 64)}
    if op == "batch":
        return {"op": op, "images": rng.randint(4, 48), "lo": rng.randint(128, 256),
                "hi": rng.randint(512, 2048), "mode": rng.choice(["ref", "std"])}
    if op == "inplace":
        r = rng.choice([2, 3, 5, 7, 9])
        return {"op": op, "w": _size(rng, 128, 2048), "h": _size(rng, 128, 2048), "r": r,
                "mode": rng.choice(["ref", "std"]), "ss": round(max(0.7, r / 1.5), 3),
                "sr": round(rng.uniform(10.0, 50.0), 3), "noise": noise,
                "repeat": rng.randint(1, 4)}
    if op == "cluster":
        gap = rng.choice([10, 10, 12, 40])
        return {"op": op, "w": _size(rng, 128, 4096), "h": _size(rng, 128, 4096),
                "range": rng.choice([3, 8, 8, 16]), "count": rng.choice([5, 5, 7]), "gap": gap,
                "diffe": gap, "noise": noise}
    if op == "regions":
        return {"op": op, "w": _size(rng, 128, 4096), "h": _size(rng, 128, 4096),
                "noise": round(rng.uniform(0.5, 10.0), 2)}
    if op == "chain":
        return {"op": op, "w": _size(rng, 256, 4096), "h": _size(rng, 256, 4096), "noise": noise}
    if op == "surrogate":
        return {"op": op, "w": _size(rng, 256, 4096), "h": _size(rng, 256, 4096), "r": 15,
                "ss": 10.0, "sr": round(rng.uniform(15.0, 45.0), 3), "noise": noise}
    return {"op": "train", "n": rng.randint(4, 64), "h": rng.randint(48, 256),
            "w": rng.randint(48, 256)}


# ------------------------------------------------------------------ inputs

def _image(w, h, noise, g, r):
    """A (h, w) uint8 device image: gradient, shapes, noise (g: the device's
    noise generator, r: a numpy generator for the shapes)."""
    s = math.sqrt(w * h) / 512.0
    n = max(1, round(40 * s))
    lo, hi = max(1, round(8 * s ** 0.5)), max(2, round(96 * s))
    img = torch.linspace(0.0, 200.0, w, device="cuda").expand(h, w).contiguous()
    for k in range(2 * n):
        sw, sh = (int(v) for v in r.integers(lo, hi + 1, 2))
        x, y = int(r.integers(-sw // 2, w)), int(r.integers(-sh // 2, h))
        grey = float(r.integers(0, 256))
        if k % 2 == 0:
            img[max(y, 0):max(y + sh, 0), max(x, 0):max(x + sw, 0)] = grey
        else:
            rad = sw / 2
            y0, y1 = max(int(y - rad), 0), min(int(y + rad) + 1, h)
            x0, x1 = max(int(x - rad), 0), min(int(x + rad) + 1, w)
            if y0 >= y1 or x0 >= x1:
                continue
            yy = torch.arange(y0, y1, device="cuda", dtype=torch.float32)[:, None] - y
            xx = torch.arange(x0, x1, device="cuda", dtype=torch.float32)[None, :] - x
            img[y0:y1, x0:x1].masked_fill_(yy * yy + xx * xx <= rad * rad, grey)
    img += noise * torch.randn((h, w), generator=g, device="cuda")
    return img.round_().clamp_(0, 255).to(torch.uint8)


def _rngs(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed)), np.random.default_rng(int(seed))


def _mode(case):
    return oc.MODE_REF if case["mode"] == "ref" else oc.MODE_STD


def _batch_plan(case):
    """Image sizes, ROIs, radii and sigma_range of a batch (the same for every
    seed: a program's set of cameras)."""
    r = np.random.default_rng([case["images"], case["lo"], case["hi"]])
    plan = []
    for _ in range(case["images"]):
        w, h = (int(v) for v in r.integers(case["lo"], case["hi"] + 1, 2))
        rw, rh = int(r.integers((w + 1) // 2, w + 1)), int(r.integers((h + 1) // 2, h + 1))
        x, y = int(r.integers(0, w - rw + 1)), int(r.integers(0, h - rh + 1))
        plan.append((w, h, (x, y, x + rw, y + rh), (3, 5, 9)[int(r.integers(0, 3))],
                     10.0 + 40.0 * float(r.random())))
    return plan


def _initial_params(seed):
    """Flat network parameters at the start of a training run: normal weights
    of variance 2 / fan-in, the last layer at a tenth, zero biases."""
    r = np.random.default_rng([int(seed), 6])
    out = []
    for layer in range(6):
        cin, cout = (2 if layer == 0 else 32), (1 if layer == 5 else 32)
        sd = math.sqrt(2.0 / (9.0 * cin)) * (0.1 if layer == 5 else 1.0)
        out += [sd * r.standard_normal(9 * cin * cout), np.zeros(cout)]
    return np.concatenate(out).astype(np.float32)


def _weighted_mean(x, radius, ss, sr):
    """Plain torch range-and-space weighted mean of (n, h, w) bytes, whole
    greys: the training target."""
    xf = x.float()
    n, h, w = xf.shape
    p = torch.nn.functional.pad(xf[:, None], (radius,) * 4, mode="replicate")[:, 0]
    t, s = torch.zeros_like(xf), torch.zeros_like(xf)
    q = (-0.5 / (sr * sr))[:, None, None]
    for dy in range(-radius, radius + 1):
        for dx in range(-radius, radius + 1):
            v = p[:, radius + dy:radius + dy + h, radius + dx:radius + dx + w]
            f = torch.exp((v - xf) ** 2 * q) * math.exp(-(dy * dy + dx * dx) / (2.0 * ss * ss))
            t += f * v
            s += f
    return (t / s).to(torch.uint8)


def _train_inputs(case, seed):
    """Crops, targets, sigma_range and edge bits of one batch."""
    g, r = _rngs(seed)
    n, h, w = case["n"], case["h"], case["w"]
    big = _image(max(4 * w, 512), max(4 * h, 512), 12.0, g, r)
    x = torch.empty((n, h, w), dtype=torch.uint8, device="cuda")
    for i in range(n):
        oy, ox = int(r.integers(0, big.shape[0] - h + 1)), int(r.integers(0, big.shape[1] - w + 1))
        x[i] = big[oy:oy + h, ox:ox + w]
    sigma = torch.from_numpy(r.uniform(15.0, 45.0, n).astype(np.float32)).cuda()
    y = _weighted_mean(x, 5, 10.0, sigma)
    edges = torch.from_numpy((r.integers(0, 16, n) * (r.random(n) < 0.4)).astype(np.uint8)).cuda()
    return x, y, sigma, edges


def _roi(case):
    px, py = case.get("pad_x", 0), case.get("pad_y", 0)
    x, y = px // 3, py // 2
    return (x, y, x + case["w"], y + case["h"])


def prepare(case, seed):
    op = case["op"]
    g, r = _rngs(seed)
    st = {"case": case, "op": op}
    if op == "train":
        st["net"] = sg.Surrogate(seed=1)
        st["net"].set_params(_initial_params(seed))
        st["x"], st["y"], st["sigma"], st["edges"] = _train_inputs(case, seed)
        return st
    if op == "batch":
        st["in"], st["out"], st["lut"], jobs = [], [], [], []
        for w, h, roi, rad, sr in _batch_plan(case):
            st["in"].append(_image(w, h, 10.0, g, r))
            st["out"].append(torch.zeros((roi[3] - roi[1], roi[2] - roi[0]), dtype=torch.uint8,
                                         device="cuda"))
            st["lut"].append(oc.Lut.from_sigmas(rad / 1.5, sr))
            jobs.append(oc.Job(oc.view(st["in"][-1], roi), oc.view(st["out"][-1]),
                               st["lut"][-1].handle, rad, _mode(case)))
        st["batch"] = oc.Batch(jobs)
        return st
    w, h = case["w"], case["h"]
    st["img"] = _image(w + case.get("pad_x", 0), h + case.get("pad_y", 0), case["noise"], g, r)
    st["roi"] = _roi(case)
    st["out"] = torch.zeros((h, w), dtype=torch.uint8, device="cuda")
    if op in ("filter", "inplace", "surrogate"):
        st["lut"] = oc.Lut.from_sigmas(case["ss"], case["sr"])
    if op == "inplace":
        st["work"] = torch.empty(h * w, dtype=torch.uint8, device="cuda")
    if op == "chain":
        st["lut"] = oc.Lut.from_sigmas(5.0, 25.0)
        st["lc"], st["bf"] = torch.zeros_like(st["out"]), torch.zeros_like(st["out"])
    if op == "surrogate":
        st["net"] = sg.Surrogate(seed=1)
        st["net"].load(sg.DEFAULT_WEIGHTS)
    return st


def run(state):
    case, op = state["case"], state["op"]
    if op == "filter":
        oc.exact(oc.view(state["img"], state["roi"]), oc.view(state["out"]), state["lut"],
                 case["r"], _mode(case))
        return state["out"]
    if op == "batch":
        state["batch"].run_graph()
        return state["out"]
    if op == "inplace":
        # the frame arrives in the buffer that is filtered in place
        state["out"].copy_(state["img"])
        oc.exact_inplace(oc.view(state["out"]), state["lut"], case["r"], _mode(case),
                         repeat=case["repeat"], work=state["work"])
        return state["out"]
    if op == "cluster":
        oc.local_cluster(oc.view(state["img"]), oc.view(state["out"]), case["range"],
                         case["count"], case["gap"], case["diffe"])
        return state["out"]
    if op == "regions":
        oc.connect_region(oc.view(state["img"]), oc.view(state["out"]))
        return state["out"]
    if op == "chain":
        oc.local_cluster(oc.view(state["img"]), oc.view(state["lc"]))
        oc.exact(oc.view(state["lc"]), oc.view(state["bf"]), state["lut"], 7, oc.MODE_REF)
        oc.connect_region(oc.view(state["bf"]), oc.view(state["out"]))
        return [state["lc"], state["bf"], state["out"]]
    if op == "surrogate":
        state["net"].filter(oc.view(state["img"]), oc.view(state["out"]), state["lut"], case["r"],
                            oc.MODE_STD, case["sr"], 2, counts=False)
        return state["out"]
    pred, grads, loss = state["net"].forward_backward(state["x"], state["y"], state["sigma"],
                                                      edges=state["edges"])
    return {"pred": pred, "grads": grads, "loss": loss}


def _taps(r, mode):
    return (2 * r + 1) ** 2 + (1 if mode == "ref" else 0)


def work(case):
    op = case["op"]
    if op == "train":
        px = case["n"] * case["h"] * case["w"]
        # bytes in, the prediction and the gradients out; forward, data and
        # weight gradients are one product of the network's size each
        return {"bytes": 2 * px + 4 * px + 8 * NET_PARAMS, "flops": 3 * NET_FLOP * px}
    if op == "batch":
        px = [((roi[2] - roi[0]) * (roi[3] - roi[1]), rad)
              for _, _, roi, rad, _ in _batch_plan(case)]
        return {"bytes": sum(2 * p for p, _ in px),
                "flops": sum(p * (4 * _taps(rad, case["mode"]) + 1) for p, rad in px)}
    px = case["w"] * case["h"]
    if op == "filter":
        return {"bytes": 2 * px, "flops": px * (4 * _taps(case["r"], case["mode"]) + 1)}
    if op == "inplace":
        n = case["repeat"]
        return {"bytes": 2 * px * (n + 1), "flops": n * px * (4 * _taps(case["r"], case["mode"]) + 1)}
    if op == "cluster":
        # per direction one gap and one side test, then the mean of 8 averages
        return {"bytes": 2 * px, "flops": 64 * px}
    if op == "regions":
        return {"bytes": 2 * px, "flops": 8 * px}
    if op == "chain":
        return {"bytes": 6 * px, "flops": px * (72 + 4 * _taps(7, "ref") + 1)}
    # the network and the exact samples (1 in 64 pixels)
    return {"bytes": 2 * px, "flops": px * (NET_FLOP + (4 * _taps(case["r"], "std") + 1) / 64)}


# ------------------------------------------------------------- 64-bit values

def _layers(params):
    """[(W[9][cin][cout], b[cout])] in double from the flat parameters."""
    out, at = [], 0
    for layer in range(6):
        cin, cout = (2 if layer == 0 else 32), (1 if layer == 5 else 32)
        w = params[at:at + 9 * cin * cout].reshape(9, cin, cout)
        at += 9 * cin * cout
        out.append((w, params[at:at + cout]))
        at += cout
    return out


def _conv(x, w, b):
    """3x3 zero-padded convolution of (n, h, w, cin) as nine products."""
    n, h, wd, cin = x.shape
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    acc = b
    for t in range(9):
        s = p[:, t // 3:t // 3 + h, t % 3:t % 3 + wd].reshape(-1, cin)
        acc = acc + s @ w[t]
    return acc.reshape(n, h, wd, -1)


def exact(case, seed):
    """Double-precision prediction, gradients and loss of a training pass.
    Every other case returns bytes, which are whole numbers."""
    if case["op"] != "train":
        return None
    x, y, sigma, edges = _train_inputs(case, seed)
    n, h, w = x.shape
    params = torch.from_numpy(_initial_params(seed).astype(np.float64)).cuda().requires_grad_(True)
    m = CROP_MARGIN
    count = n * (h - 2 * m) * (w - 2 * m)
    preds, loss = [], 0.0
    for i in range(0, n, 8):
        u = x[i:i + 8].double() / 255.0
        a = torch.stack([u, (sigma[i:i + 8].double() / 100.0)[:, None, None].expand_as(u)], -1)
        layers = _layers(params)
        for k, (wt, b) in enumerate(layers):
            a = _conv(a, wt, b)
            if k < 5:
                a = a.relu()
        p = u + a[..., 0]
        e = edges[i:i + 8].to(torch.int64)[:, None, None]
        yy = torch.arange(h, device="cuda")[None, :, None]
        xx = torch.arange(w, device="cuda")[None, None, :]
        keep = (((yy >= m) | (e & 1 > 0)) & ((yy < h - m) | (e & 2 > 0)) &
                ((xx >= m) | (e & 4 > 0)) & ((xx < w - m) | (e & 8 > 0)))
        d = (p - y[i:i + 8].double() / 255.0) * keep
        part = (d * d).sum() / count
        part.backward()
        loss += float(part.detach())
        preds.append(p.detach())
    return {"pred": torch.cat(preds), "grads": params.grad,
            "loss": torch.tensor([loss], dtype=torch.float64, device="cuda")}
