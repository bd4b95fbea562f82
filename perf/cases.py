"""Performance cases: what a user of this library has it do, from the smallest call to the largest.

A case is a compiled network (or a single layer) at one image extent, run through one of the library's entry points:

  device   `Instance.infer_device` on tensors that live in GPU memory (a renderer's frame buffers)
  host     `Module.__call__` on a numpy array: upload, dispatches and download in one blocking call
  stream   `Instance.infer_many` on a sequence of frames in page-locked host memory

Networks are those of `denox_amd.networks` with their seeded weights; "conv" is one convolution with its activation, "layers" the
data-movement layers (pad, pool, upsample, concat, activation, crop) without a convolution that could absorb them.  A network is
compiled as `compile_model` does it by default (schedule from estimates) or, where a case says so, against a timing table measured
on the GPU first (`Db.populate`, `Db.bench`), the workflow of the benchmark.
"""
import functools
import os
import tempfile

import numpy as np
import torch

import denox_amd as dx
from denox_amd import networks


def _unet(name, H, W, **kw):
    return {"name": name, "net": "oidn_unet", "mult": 1, "H": H, "W": W, "layout": "HWC", "entry": "device", "tuned": False, **kw}


def _conv(name, C, K, H, W, **kw):
    return {"name": name, "net": "conv", "C": C, "K": K, "R": 3, "stride": 1, "act": "relu", "H": H, "W": W, "layout": "HWC", "entry": "device", "tuned": False, **kw}


def _layers(name, C, H, W, **kw):
    return {"name": name, "net": "layers", "C": C, "pool": "max", "H": H, "W": W, "layout": "HWC", "entry": "device", "tuned": False, **kw}


def listed():
    return [
        # the smallest network call: six layers on a thumbnail, nothing but launches and latency
        {"name": "tiny_128", "net": "tiny_unet", "H": 128, "W": 128, "layout": "HWC", "entry": "device", "tuned": False},
        # a preview or one tile of a tiled render, ragged extents (padded to multiples of 16 inside the network)
        _unet("unet_187x251", 187, 251),
        # the denoising U-Net at the usual video extent, compiled without tuning
        _unet("unet_1080p", 1080, 1920),
        # ... and with the schedule tuned on this GPU: the benchmark's headline
        _unet("unet_1080p_tuned", 1080, 1920, tuned=True),
        # the largest frame of the benchmark
        _unet("unet_4k", 2160, 3840),
        # doubled widths, planar interface, odd extents
        _unet("unet2x_chw_1077", 1077, 1917, mult=2, layout="CHW"),
        # host arrays in and out, one blocking call per frame (a script that denoises images)
        _unet("host_1080p", 1080, 1920, entry="host"),
        # a sequence of frames from page-locked memory (video)
        _unet("stream_720p", 720, 1280, entry="stream"),
        # one wide full-resolution layer
        _conv("conv64_1080p", 64, 64, 1080, 1920),
        # a deep layer on a small image in the block-major layout, as the reference's own layer tests have it
        _conv("conv256_100_chwc8", 256, 256, 100, 100, layout="CHWC8", act="none"),
        # strided 5 x 5 downsampling with a leaky activation
        _conv("conv5s2_1080p", 32, 64, 1080, 1920, R=5, stride=2, act="leaky_relu"),
        # the bandwidth kernels on 9-channel pixels (colour, albedo, normals) with odd extents
        _layers("layers9_1077", 9, 1077, 1917),
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["unet", "unet", "unet", "tiny", "conv", "conv", "layers", "layers", "host", "stream", "tuned"])
    if kind == "tiny":
        return {"net": "tiny_unet", "H": 2 * _log_uniform(rng, 32, 540), "W": 2 * _log_uniform(rng, 32, 960), "layout": rng.choice(["HWC", "CHW"]), "entry": "device", "tuned": False}
    if kind == "conv":
        c = _conv("", rng.choice([3, 9, 16, 32, 48, 64, 80, 96, 128, 256]), rng.choice([3, 16, 32, 48, 64, 96, 128, 256]), _log_uniform(rng, 64, 1088), _log_uniform(rng, 64, 1920),
                  R=rng.choice([1, 3, 3, 3, 5]), stride=rng.choice([1, 1, 2]), act=rng.choice(["none", "relu", "leaky_relu"]),
                  layout=rng.choice(["HWC", "HWC", "CHW"]))
        while work(c)["flops"] > 1e12:  # stay below the largest listed case
            c["H"], c["W"] = (c["H"] + 1) // 2, (c["W"] + 1) // 2
    elif kind == "layers":
        c = _layers("", rng.choice([3, 8, 9, 24, 32, 64, 73]), 2 * _log_uniform(rng, 64, 1080), 2 * _log_uniform(rng, 64, 1920), pool=rng.choice(["max", "avg"]))
        c["H"] -= rng.randrange(2)
        c["W"] -= rng.randrange(2)
    elif kind == "unet":
        mult = rng.choice([1, 1, 2])
        c = _unet("", _log_uniform(rng, 96, 2160 // mult), _log_uniform(rng, 96, 3840 // mult), mult=mult, layout=rng.choice(["HWC", "HWC", "CHW"]))
    elif kind == "tuned":
        c = _unet("", _log_uniform(rng, 270, 1080), _log_uniform(rng, 480, 1920), tuned=True)
    else:
        c = _unet("", _log_uniform(rng, 128, 1080), _log_uniform(rng, 128, 1920), entry=kind)
    c.pop("name")
    return c


STREAM_FRAMES = 6


def _channels(case):
    return {"tiny_unet": 3, "oidn_unet": 9}.get(case["net"]) or case["C"]


def _network(case):
    if case["net"] == "oidn_unet":
        return networks.build("oidn_unet", width_mult=case["mult"])[0]
    if case["net"] == "tiny_unet":
        return networks.build("tiny_unet")[0]
    m = dx.Model()
    x = m.input("input", "W", "H", case["C"])
    if case["net"] == "conv":
        rng = np.random.default_rng(0)
        C, K, R, s = case["C"], case["K"], case["R"], case["stride"]
        w = (rng.standard_normal((K, C, R, R)) * np.sqrt(2.0 / (R * R * C))).astype(np.float16)
        y = m.conv2d(x, w, (rng.standard_normal(K) * 0.01).astype(np.float16), stride=(s, s), padding=(R // 2, R // 2))
        if case["act"] != "none":
            y = m.activation(y, case["act"], 0.1)
    else:
        p = m.pad_to_multiple(x, 2)
        y = m.concat(m.upsample(m.pool(p, func=case["pool"])), p)
        y = m.slice(m.activation(y, "leaky_relu", 0.1), 0, x.width, 0, x.height)
    m.output(y, "output")
    return m


@functools.lru_cache(maxsize=None)
def _compiled(key):
    """The serialised model, compiled once per process: a program loads its compiled network and keeps it."""
    case = dict(key)
    model, lay = _network(case), dx.Layout[case["layout"]]
    at = dict(assume={"H": case["H"], "W": case["W"]}, input_layout=lay, output_layout=lay)
    if not case["tuned"]:
        return dx.compile_model(model, **at)
    db = dx.Db(os.path.join(tempfile.mkdtemp(prefix="perf_cases_"), "gpu.db"))
    db.populate(model, **at)
    db.bench(min_samples=10, max_relative_error=0.03, max_samples=50, save_progress=False)
    return dx.compile_model(model, db=db, **at)


def _frame(case, seed):
    """One input frame in HWC on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    H, W, C = case["H"], case["W"], _channels(case)
    if case["net"] == "oidn_unet":  # colour (lognormal, clamped), albedo, unit normals
        color = torch.randn(H, W, 3, device="cuda", generator=g).exp().clamp(0.0, 64.0)
        albedo = torch.rand(H, W, 3, device="cuda", generator=g)
        n = torch.rand(H, W, 3, device="cuda", generator=g) * 2.0 - 1.0
        n = n / n.norm(dim=2, keepdim=True).clamp_min(1e-6)
        return torch.cat([color, albedo, n], dim=2).half()
    if case["net"] == "tiny_unet":
        return torch.rand(H, W, C, device="cuda", generator=g).half()
    x = torch.randn(H, W, C, device="cuda", generator=g)
    return (x.abs() if case["net"] == "conv" else x).half()


def _in_layout(x, layout):
    if layout == "CHW":
        return x.permute(2, 0, 1).contiguous()
    if layout == "CHWC8":
        return x.reshape(x.shape[0], x.shape[1], -1, 8).permute(2, 0, 1, 3).contiguous()
    return x


def prepare(case, seed):
    module = dx.Module.load(_compiled(tuple(sorted((k, v) for k, v in case.items() if k != "name"))))
    extents = {"H": case["H"], "W": case["W"]}
    state = {"entry": case["entry"], "module": module, "extents": extents, "instance": module.instance(**extents)}
    if case["entry"] == "stream":
        frames = [_in_layout(_frame(case, seed * STREAM_FRAMES + f), case["layout"]).cpu().numpy() for f in range(STREAM_FRAMES)]
        d = state["instance"].output_desc()
        state["frames"] = [[dx.pinned_empty(x.shape)] for x in frames]
        state["results"] = [[dx.pinned_empty((d["height"], d["width"], d["channels"]))] for _ in frames]
        for p, x in zip(state["frames"], frames):
            p[0][...] = x
        return state
    x = _in_layout(_frame(case, seed), case["layout"])
    if case["entry"] == "host":
        state["x"] = x.cpu().numpy()
    else:
        state["x"] = x
        state["y"] = torch.empty(state["instance"].output_desc()["byte_size"] // 2, dtype=torch.float16, device="cuda")
    return state


def run(state):
    if state["entry"] == "host":
        return state["module"](state["x"], **state["extents"])
    if state["entry"] == "stream":
        return [r[0] for r in state["instance"].infer_many(state["frames"], state["results"])]
    state["instance"].infer_device([state["x"].data_ptr()], [state["y"].data_ptr()])
    return state["y"]


def work(case):
    """The layers' own multiplications, and the interface tensors and weights once each."""
    H, W = case["H"], case["W"]
    model = _network(case)
    shape = {"input": (H, W, _channels(case))}
    flops = weights = 0
    for op in model.to_ops({"H": H, "W": W}):
        src = op["src"] if isinstance(op["src"], str) else op["src"][0]
        h, w, c = shape[src]
        kind = op["op"]
        if kind == "conv2d":
            K, C, R, S = op["weight"].shape
            (sy, sx), (py, px) = op["stride"], op["padding"]
            h, w, c = (h + 2 * py - R) // sy + 1, (w + 2 * px - S) // sx + 1, K
            flops += 2 * R * S * C * K * h * w
            weights += 2 * (R * S * C * K + K)
        elif kind == "pool":
            h, w = h // op["kernel"][0], w // op["kernel"][1]
        elif kind == "upsample":
            h, w = h * op["factor"], w * op["factor"]
        elif kind == "concat":
            c += shape[op["src"][1]][2]
        elif kind == "pad":
            h, w = h + op["top"] + op["bottom"], w + op["left"] + op["right"]
        elif kind == "slice":
            h, w = op["out_h"], op["out_w"]
        shape[op["dst"]] = (h, w, c)
    frames = STREAM_FRAMES if case["entry"] == "stream" else 1
    h, w, c = shape[model.outputs[0].name]
    return {"bytes": frames * 2 * (H * W * _channels(case) + h * w * c) + weights, "flops": frames * flops}


def tolerance(case):
    # Data movement and element-wise binary16 arithmetic: the same bits.  Convolutions accumulate in binary32 and round every layer's
    # result to binary16 once; kernels differ in summation order and in whether coinciding taps of an upsampled source are summed (and
    # rounded) beforehand.  Measured between kernels of different order: one layer 1e-5 in norm and one unit in the last place, the
    # four-layer network a few times that, sixteen layers of lognormal input 1.4e-3 / 9e-3; four times as much is allowed.
    if case["net"] == "layers":
        return "exact"
    if case["net"] == "conv":
        return {"rel": 5e-5, "max": 4e-3}
    return {"rel": 6e-3, "max": 0.04} if case["net"] == "oidn_unet" else {"rel": 2e-4, "max": 8e-3}


def exact(case, seed):
    """The layers one after the other in binary64 with torch; every output value in the order `run` returns it."""
    if case["entry"] == "stream":
        return [_exact_frame(case, seed * STREAM_FRAMES + f) for f in range(STREAM_FRAMES)]
    return _exact_frame(case, seed)


def _exact_frame(case, seed):
    model = _network(case)
    t = {"input": _frame(case, seed).permute(2, 0, 1).double()}
    ops = model.to_ops({"H": case["H"], "W": case["W"]})
    last = {s: i for i, op in enumerate(ops) for s in ([op["src"]] if isinstance(op["src"], str) else op["src"])}
    for i, op in enumerate(ops):
        names = [op["src"]] if isinstance(op["src"], str) else op["src"]
        x, kind = t[names[0]], op["op"]
        if kind == "conv2d":
            w = torch.from_numpy(np.asarray(op["weight"])).cuda().double()
            b = torch.from_numpy(np.asarray(op["bias"])).cuda().double()
            (sy, sx), (py, px) = op["stride"], op["padding"]
            K, C, R, S = w.shape
            xp = torch.nn.functional.pad(x, (px, px, py, py))
            h, wd = (x.shape[1] + 2 * py - R) // sy + 1, (x.shape[2] + 2 * px - S) // sx + 1
            y = b[:, None].expand(K, h * wd).contiguous()
            for r in range(R):
                for s in range(S):
                    y.addmm_(w[:, :, r, s].contiguous(), xp[:, r:r + (h - 1) * sy + 1:sy, s:s + (wd - 1) * sx + 1:sx].reshape(C, h * wd))
            y = y.view(K, h, wd)
        elif kind == "activation":
            # the slope is a binary16 number, and these networks apply it to binary16 values
            y = x.clamp_min(0.0) if op["func"] == "relu" else torch.where(x > 0, x, x * float(np.float16(op["alpha"])))
        elif kind == "pool":
            n = x.reshape(x.shape[0], x.shape[1] // 2, 2, x.shape[2] // 2, 2)
            y = n.amax(dim=(2, 4)) if op["func"] == "max" else n.mean(dim=(2, 4))
        elif kind == "upsample":
            y = x.repeat_interleave(op["factor"], 1).repeat_interleave(op["factor"], 2)
        elif kind == "concat":
            y = torch.cat([x, t[names[1]]])
        elif kind == "pad":
            y = torch.nn.functional.pad(x[None], (op["left"], op["right"], op["top"], op["bottom"]), mode="replicate")[0]
        elif kind == "slice":
            y = x[:, op["top"]:op["top"] + op["out_h"], op["left"]:op["left"] + op["out_w"]]
        for s in set(names):
            if last[s] == i:
                del t[s]
        t[op["dst"]] = y
    y = t[model.outputs[0].name]
    if case["layout"] == "HWC":
        y = y.permute(1, 2, 0)
    elif case["layout"] == "CHWC8":
        y = y.reshape(-1, 8, *y.shape[1:]).permute(0, 2, 3, 1)
    y = y.contiguous()
    return y.reshape(-1) if case["entry"] == "device" else y.cpu().numpy()
