#!/usr/bin/env python3
"""Headline benchmark: OIDN-style 9->3 U-Net, fp16 HWC, 1920x1080, one MI355X.

A "step" is one whole-network inference of one synthetic frame that is already
resident in HBM (device pointers in, device pointer out), launched through the
C ABI (denox_hip_instance_infer_device) on the library's stream: one hipGraph, or plain
launches where the schedule has at most four dispatches.

Prints ONE JSON line: Mpix/s (= 1920*1080 / time per frame) with ms/frame in
`ms_per_step`, a `roofline` object for the dominant kernel (per-dispatch
hipEvent timing on the launch stream), a `cpu_baseline` object (the CPU oracle
timed on one frame of the same workload) and a `parity` object: the output of
the schedule that was just timed against that oracle frame (exit status 1 when
it misses the bar).
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_FP16_MFMA_TFLOPS = 2500.0  # MI355X dense fp16, published
PEAK_HBM_GBPS = 8000.0          # MI355X HBM3E, published


# name -> (network, builder kwargs, H, W, interface layout, description)
WORKLOADS = {
    "tiny_128": ("tiny_unet", {}, 128, 128, "HWC", "tiny 2-level U-Net 3->3, fp16 HWC, 128x128"),
    "conv64_1080p": ("single_conv", {}, 1080, 1920, "HWC", "conv3x3 64->64 + bias + ReLU, fp16 HWC, 1920x1080"),
    "oidn_1080p": ("oidn_unet", {}, 1080, 1920, "HWC", "OIDN-style U-Net 9->3, fp16 HWC, 1920x1080, replicate-pad to multiple of 16 + crop included"),
    "oidn_4k": ("oidn_unet", {}, 2160, 3840, "HWC", "OIDN-style U-Net 9->3, fp16 HWC, 3840x2160"),
    "oidn2x_chw_1077": ("oidn_unet", {"width_mult": 2}, 1077, 1917, "CHW",
                        "OIDN-style U-Net with doubled widths 9->3, fp16, CHW in/out, 1917x1077, replicate-pad to 1920x1088 + crop included"),
}


OTHER_WORKLOADS = ["conv64_1080p", "oidn_4k", "oidn2x_chw_1077"]  # printed beside the headline, briefly
OTHER_STEPS, OTHER_WARMUP = 30, 5


def lavapipe_probe() -> str:
    """The reference's own CPU route (its SPIR-V on Mesa lavapipe) needs a Vulkan loader, the
    lavapipe ICD and a built denox; report why it is unavailable rather than inventing a number."""
    import ctypes.util
    if ctypes.util.find_library("vulkan") is None:
        return "unavailable (no Vulkan loader on this machine)"
    if ctypes.util.find_library("vulkan_lvp") is None:
        return "unavailable (no lavapipe ICD on this machine)"
    return "unavailable (denox itself cannot be built here: needs glslang, SPIRV-Tools, FlatBuffers)"


def parity_object(r: dict, pixels: int, against: str) -> dict:
    """`oracle.conv_parity`'s verdict as it is printed: the errors, the stated bar's own verdict, the floor and the bar in force."""
    return {"max_abs": r["max_abs"], "mean_abs": r["mean_abs"], "stated_bar": [2e-2, 2e-3], "meets_stated_bar": r["literal_ok"],
            "floor_max_abs": r["floor_max_abs"], "floor_mean_abs": r["floor_mean_abs"],
            "floor": "error of the oracle's binary16-storage evaluation (fp32 accumulation, one rounding per layer) against its fp32 evaluation "
                     "(null: not evaluated, the stated bar was met)",
            "bar_max_abs": r["bar_max_abs"], "bar_mean_abs": r["bar_mean_abs"],
            "bar": f"max(stated, {oracle_factor('max')} x floor max) / max(stated, {oracle_factor('mean')} x floor mean)",
            "pixels_compared": pixels, "against": against, "ok": r["ok"]}


def oracle_factor(which: str) -> float:
    import oracle
    return oracle.FLOOR_FACTOR_MAX if which == "max" else oracle.FLOOR_FACTOR_MEAN


def crop_parity(net: str, kw: dict, seed: int, H: int, W: int, gpu_out_hwc, spots, size: int = 272) -> dict:
    """The timed schedule's output against the oracle on 16-aligned crops of the same frame: a crop's evaluation equals the
    full frame's `margin` pixels inside every cut edge (the receptive field of the deepest network here is below 96 pixels;
    a single 3x3 conv needs 1).  Used for the workloads printed beside the headline, where a whole-frame CPU evaluation would
    take minutes."""
    import numpy as np
    import oracle
    from denox_amd import networks
    oracle.build()
    model, _ = networks.build(net, seed=seed, **kw)
    x = networks.synthetic_input(net, H, W, seed=seed)
    margin = 96 if net == "oidn_unet" else 16
    name = model.outputs[0].name
    got, want, floors = [], [], []
    for y0, x0 in spots:
        y0, x0 = y0 - y0 % 16, x0 - x0 % 16
        h, w = min(size, H - y0), min(size, W - x0)
        crop = np.ascontiguousarray(x[y0:y0 + h, x0:x0 + w])
        ops = model.to_ops({"H": h, "W": w})
        ys = slice(0 if y0 == 0 else margin, h if y0 + h >= H else h - margin)
        xs = slice(0 if x0 == 0 else margin, w if x0 + w >= W else w - margin)
        want.append(oracle.run_graph(ops, {"input": crop}, "fp32")[name][ys, xs].reshape(-1))
        floors.append(oracle.run_graph(ops, {"input": crop}, "f16")[name][ys, xs].reshape(-1))
        got.append(np.asarray(gpu_out_hwc[y0:y0 + h, x0:x0 + w][ys, xs]).reshape(-1))
    got, want, floors = np.concatenate(got), np.concatenate(want), np.concatenate(floors)
    return parity_object(oracle.conv_parity(got, want, floors), int(got.size // gpu_out_hwc.shape[2]),
                         f"CPU oracle, fp32 evaluation of {len(spots)} crops of {size}x{size} of the same frame, compared {margin} pixels inside every cut edge")


def cpu_baseline(net: str, kw: dict, seed: int, H: int, W: int, gpu_out_hwc) -> dict:
    """CPU oracle (fp32 evaluation, OpenMP over rows) on one frame of the workload, same network, weights and input
    (the top-left 1920 x 1080 window of larger frames, 16-aligned), timed as the CPU baseline -- and, since it is the fp32
    evaluation the parity bar is defined against, compared with what the GPU schedule just timed has produced."""
    import numpy as np
    import oracle
    from denox_amd import networks
    oracle.build()
    budget_h, budget_w = (H if H <= 1088 else 1072), (W if W <= 1920 else 1920)
    model, _ = networks.build(net, seed=seed, **kw)
    x = np.ascontiguousarray(networks.synthetic_input(net, H, W, seed=seed)[:budget_h, :budget_w])
    ops = model.to_ops({"H": budget_h, "W": budget_w})
    t0 = time.perf_counter()
    want = oracle.run_graph(ops, {"input": x}, "fp32")[model.outputs[0].name]
    dt = time.perf_counter() - t0
    # A window cut out of a larger frame equals the frame's result only away from the cut: the deepest network here sees
    # less than 96 pixels in each direction.
    ys = slice(0, budget_h if budget_h == H else budget_h - 96)
    xs = slice(0, budget_w if budget_w == W else budget_w - 96)
    got = gpu_out_hwc[:budget_h, :budget_w][ys, xs]
    # The stated bar is absolute (2e-2 / 2e-3).  Where outputs are large enough that storing every tensor as binary16 already
    # costs more than that, the bar is a small multiple of that unavoidable error: the oracle's evaluation with binary16
    # tensors between the layers (fp32 accumulation, one rounding per layer) against its fp32 evaluation.
    def floor():
        return oracle.run_graph(ops, {"input": x}, "f16")[model.outputs[0].name][ys, xs]
    parity = parity_object(oracle.conv_parity(got, np.asarray(want, np.float32)[ys, xs], floor), int(got.shape[0] * got.shape[1]),
                           "CPU oracle, fp32 evaluation of the same frame")
    out = {"value": budget_h * budget_w / dt * 1e-6, "unit": "Mpix/s", "cores": oracle.num_threads(), "kind": "port",
           "sample": f"one {budget_w}x{budget_h} frame of the same network, fp32 evaluation, {dt:.1f} s wall",
           "lavapipe_baseline": lavapipe_probe(), "parity": parity}
    try:
        out.update(torch_cpu_baseline(ops, x, budget_h, budget_w))
    except Exception as e:  # context only: never fail the benchmark over it
        out["torch_fp32_Mpix_s"] = None
        out["torch_error"] = str(e)[:200]
    return out


def torch_cpu_baseline(ops, x, h, w) -> dict:
    """The same frame through torch.nn.functional in fp32 on the host cores: a library evaluation for context beside
    the oracle's time (the reference's own tests compare against torch, test/system)."""
    import numpy as np
    import torch
    import torch.nn.functional as F
    env = {"input": torch.from_numpy(np.ascontiguousarray(x.astype(np.float32).transpose(2, 0, 1)))[None]}
    prepared = []
    for op in ops:
        o = dict(op)
        if o["op"] == "conv2d":
            o["weight"] = torch.from_numpy(o["weight"].astype(np.float32))
            o["bias"] = None if o.get("bias") is None else torch.from_numpy(o["bias"].astype(np.float32))
        prepared.append(o)
    t0 = time.perf_counter()
    with torch.no_grad():
        for o in prepared:
            k, src = o["op"], o["src"]
            if k == "conv2d":
                y = F.conv2d(env[src], o["weight"], o["bias"], stride=o.get("stride", (1, 1)), padding=o.get("padding", (1, 1)))
            elif k == "activation":
                y = F.relu(env[src]) if o["func"] == "relu" else F.leaky_relu(env[src], o.get("alpha", 0.0))
            elif k == "pool":
                y = F.max_pool2d(env[src], o.get("kernel", (2, 2)))
            elif k == "upsample":
                y = F.interpolate(env[src], scale_factor=o.get("factor", 2), mode="nearest")
            elif k == "concat":
                y = torch.cat([env[src[0]], env[src[1]]], 1)
            elif k == "pad":
                y = F.pad(env[src], (o["left"], o["right"], o["top"], o["bottom"]), mode="replicate")
            elif k == "slice":
                y = env[src][:, :, o["top"]:o["top"] + o["out_h"], o["left"]:o["left"] + o["out_w"]]
            else:
                raise ValueError(k)
            env[o["dst"]] = y
    dt = time.perf_counter() - t0
    return {"torch_fp32_Mpix_s": h * w / dt * 1e-6, "torch_threads": torch.get_num_threads(), "torch_seconds": round(dt, 2)}


def measure(args, workload: str, steps: int, warmup: int, brief: bool):
    """One workload: tune, compile, time `steps` inferences after `warmup`, describe the longest dispatch, check the output.
    `brief` (the workloads printed beside the headline): fewer timing samples per candidate, no host-pointer paths, no unfused
    second schedule, parity on crops instead of the whole frame.  Returns (JSON object, exit status)."""
    import numpy as np
    import torch
    import denox_amd as dx
    from denox_amd import networks

    net, net_kw, H, W, layout, description = WORKLOADS[workload]
    if not brief:
        H, W = args.height or H, args.width or W
    model, _ = networks.build(net, seed=args.seed, **net_kw)
    lay = dx.Layout[layout]
    # The reference workflow: populate the table with every candidate dispatch, time them on
    # this GPU, then compile against the measured latencies (README.md:112-199 of the reference:
    # `denox populate`, `denox bench`, `denox compile --db`).
    features = dict(layout_preference=args.layout_preference, blocked_layout=not args.no_blocked_layout, upsample_fold=not args.no_upsample_fold)
    db = None
    tune_s = 0.0
    if not args.no_tune:
        import tempfile
        t0 = time.perf_counter()
        db = dx.Db((args.db if not brief else None) or os.path.join(tempfile.mkdtemp(prefix="denox_hip_"), "gpu.db"))
        db.populate(model, assume={"H": H, "W": W}, conv_config=args.conv_config, input_layout=lay, output_layout=lay, features=features)
        if brief:
            db.bench(min_samples=5, max_relative_error=0.05, max_samples=20)
        else:
            db.bench(min_samples=10, max_relative_error=0.03, max_samples=50, save_progress=bool(args.db))
        tune_s = time.perf_counter() - t0
    blob = dx.compile_model(model, assume={"H": H, "W": W}, conv_config=args.conv_config, db=db, input_layout=lay, output_layout=lay,
                            features=features)
    report = dx.last_compile_report()
    if args.per_dispatch:
        print(report, file=sys.stderr)
    mod = dx.Module.load(blob)
    inst = mod.instance(H=H, W=W)

    x = networks.synthetic_input(net, H, W, seed=args.seed)
    if layout == "CHW":
        x = np.ascontiguousarray(x.transpose(2, 0, 1))
    d_in = torch.from_numpy(x).cuda()
    d_out = torch.empty(inst.output_desc()["byte_size"] // 2, dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()
    ins, outs = [d_in.data_ptr()], [d_out.data_ptr()]

    # Untimed pre-roll: a part that has just been idle (compiling, tuning with pauses between candidates) runs its first
    # frames at a higher clock than it sustains; 0.3 s of back-to-back frames let clock and temperature settle, so that a
    # short timed region (--steps 20) measures the same state as a long one.
    t0 = time.perf_counter()
    while time.perf_counter() - t0 < args.settle_seconds:
        for _ in range(10):
            inst.infer_device(ins, outs)
        inst.synchronize()
    for _ in range(warmup):
        inst.infer_device(ins, outs)
    inst.synchronize()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        inst.infer_device(ins, outs)
    inst.synchronize()
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    ms = dt / steps * 1e3
    # single replays, each synchronised and timed on the host (launch latency included): the spread of the frame time, for
    # context; `value` is the bulk timing above.  A single replay starts on an idle part, a bulk frame follows another one.
    singles = []
    for _ in range(20 if brief else min(100, max(20, steps))):
        inst.synchronize()
        t1 = time.perf_counter()
        inst.infer_device(ins, outs)
        inst.synchronize()
        singles.append((time.perf_counter() - t1) * 1e3)
    singles.sort()
    out_host = d_out.cpu().numpy()  # what the timed schedule wrote in its last step
    if not np.isfinite(out_host).all():
        print(f"bench.py: non-finite output ({workload})", file=sys.stderr)
        return None, 1
    od = inst.output_desc()
    out_hwc = out_host.reshape(od["channels"], od["height"], od["width"]).transpose(1, 2, 0) if layout == "CHW" else out_host.reshape(od["height"], od["width"], od["channels"])

    host_ms = pipelined_ms = None
    if not brief:
        # the reference's own entry point (host pointers in and out, blocking): PCIe-inclusive, reported beside, never as `value`
        t0 = time.perf_counter()
        for _ in range(3):
            y_host = inst.infer(x)[0]
        host_ms = (time.perf_counter() - t0) / 3 * 1e3
        # the same from page-locked memory with uploads, dispatches and downloads of neighbouring frames overlapped
        # (denox_hip_instance_infer_many); reported, never `value`
        nf = 16
        pin_in = [[dx.pinned_empty(np.asarray(x).shape)] for _ in range(2)]  # two buffers a side, used in turn
        pin_out = [[dx.pinned_empty(y_host.shape)] for _ in range(2)]
        for b in pin_in:
            b[0][...] = x
        inst.infer_many(pin_in, pin_out)
        t0 = time.perf_counter()
        inst.infer_many([pin_in[f & 1] for f in range(nf)], [pin_out[f & 1] for f in range(nf)])
        pipelined_ms = (time.perf_counter() - t0) / nf * 1e3
        assert np.array_equal(pin_out[0][0], y_host) and np.array_equal(pin_out[1][0], y_host)
        del pin_in, pin_out

    # Two frames in flight: a second instance of the same compiled model in a context (a stream) of its own, both fed from
    # device memory.  The dispatches of one frame fill the launch ramps, tails and half-empty low-resolution layers of the
    # other.  A throughput figure for a stream of frames; a frame then takes about twice as long to come back, so it is
    # reported beside `value`, which stays one frame at a time.
    two_ms = None
    if not brief and not args.no_two_frames:
        ctx2 = dx.Context(0)
        mod2 = dx.Module.load(blob, ctx2)
        inst2 = mod2.instance(H=H, W=W)
        d_in2, d_out2 = d_in.clone(), torch.zeros_like(d_out)
        torch.cuda.synchronize()
        ins2, outs2 = [d_in2.data_ptr()], [d_out2.data_ptr()]
        def both(n):
            for _ in range(n):
                inst.infer_device(ins, outs)
                inst2.infer_device(ins2, outs2)
            inst.synchronize()
            inst2.synchronize()
        both(20)
        n2 = max(50, steps // 2)
        t0 = time.perf_counter()
        both(n2)
        two_ms = (time.perf_counter() - t0) / (2 * n2) * 1e3
        if not torch.equal(d_out2, d_out):
            print("bench.py: the second instance's output differs from the first's", file=sys.stderr)
            return None, 1
        del inst2, mod2, ctx2, d_in2, d_out2

    # per-dispatch hipEvent timings on the launch stream, averaged over several passes
    passes = 2 if brief else 5
    acc = None
    for _ in range(passes):
        t = inst.bench(warmup=2)
        if acc is None:
            acc = t
        else:
            for a, b in zip(acc, t):
                a["latency_ms"] += b["latency_ms"]
    for a in acc:
        a["latency_ms"] /= passes
        a["GBps"] = (a["memory_reads"] + a["memory_writes"]) / a["latency_ms"] * 1e-6
        a["TFLOPs"] = a["flops"] / a["latency_ms"] * 1e-9
    if args.per_dispatch:
        print(dx.report(acc), file=sys.stderr)
    dom = max(acc, key=lambda a: a["latency_ms"])
    conv = [a for a in acc if a["flops"] > 0 and "conv" in a["name"]]
    conv_ms = sum(a["latency_ms"] for a in conv)
    conv_flops = sum(a["flops"] for a in conv)
    other = [a for a in acc if a not in conv]
    other_ms = sum(a["latency_ms"] for a in other)
    other_bytes = sum(a["memory_reads"] + a["memory_writes"] for a in other)
    # the dominant dispatch as it runs inside the frame: events around it alone in whole inferences on the launch stream
    # (in the per-dispatch pass above every kernel repeats back to back, which a matrix-bound kernel answers with lower clocks)
    dom_ms = inst.bench_in_frame(acc.index(dom), frames=30 if brief else 100, warmup=5)
    if len(acc) == 1:
        # a schedule of one dispatch: the timed step is that dispatch and nothing else, and holds less overhead than an interval between
        # two events does
        dom_ms = min(dom_ms, ms)
    dom_tflops = dom["flops"] / dom_ms * 1e-9
    roofline = {"bound": "mfma", "kernel": dom["name"], "achieved": dom_tflops, "peak": PEAK_FP16_MFMA_TFLOPS, "unit": "TFLOP/s",
                "frac": dom_tflops / PEAK_FP16_MFMA_TFLOPS, "traffic": None,
                "kernel_ms": dom_ms, "kernel_ms_back_to_back": dom["latency_ms"],
                "kernel_GBps": (dom["memory_reads"] + dom["memory_writes"]) / dom_ms * 1e-6,
                "all_conv_TFLOPs": conv_flops / conv_ms * 1e-9 if conv_ms else None,
                "all_conv_frac": conv_flops / conv_ms * 1e-9 / PEAK_FP16_MFMA_TFLOPS if conv_ms else None,
                "non_conv_GBps": other_bytes / other_ms * 1e-6 if other_ms else None,
                "non_conv_frac_of_hbm": other_bytes / other_ms * 1e-6 / PEAK_HBM_GBPS if other_ms else None,
                "sum_dispatch_ms": sum(a["latency_ms"] for a in acc)}

    # Which configuration each dispatch of the schedule runs, and the SHA-256 of its code object.
    described = dx.describe(blob, H=H, W=W)
    desc = described["dispatches"]
    chwc8 = sum(1 for t in described["tensors"] if not t["param"] and t["format"] == 3)
    chosen = [f'{d["name"]}: {d["debug_info"].split(" | ")[0]}' for d in desc]
    dom_desc = desc[acc.index(dom)]
    roofline["kernel_entry_point"] = dom_desc["entry_point"]
    roofline["kernel_code_sha256"] = dom_desc["code_sha256"]

    if brief:
        spots = [(0, 0), (H // 2, W // 2), (H - 272 + 16, W - 272 + 16)]
        parity = None if args.no_cpu_baseline else crop_parity(net, net_kw, args.seed, H, W, out_hwc, spots)
        line = {"workload": workload, "description": description, "ms_per_step": ms, "Mpix_s": H * W / (ms * 1e-3) * 1e-6, "steps": steps, "warmup": warmup,
                "single_replay_ms_median": round(singles[len(singles) // 2], 4), "tuning_seconds": round(tune_s, 2),
                "dominant_kernel": dom_desc["entry_point"], "dominant_ms": dom_ms, "dominant_frac": roofline["frac"],
                "all_conv_frac": roofline["all_conv_frac"], "non_conv_frac_of_hbm": roofline["non_conv_frac_of_hbm"],
                "schedule_kernels": [d["entry_point"] for d in desc], "parity": parity}
        return line, (0 if parity is None or parity["ok"] else 1)

    # HBM traffic of the dominant kernel is not measured in this run: it comes from the committed rocprofv3 --pmc
    # summary, and only if that summary was taken from this very code object (same SHA-256), else null.
    roofline["traffic_source"] = "profiles/dominant_conv_traffic.json (committed rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE runs, scaled by a copy kernel of known size); not measured in this run"
    try:
        with open(os.path.join(ROOT, "profiles", "dominant_conv_traffic.json")) as f:
            tr = json.load(f)
        entry = tr["kernels"].get(dom_desc["code_sha256"])
        if entry is not None and (H, W) == (tr["height"], tr["width"]):
            roofline["traffic"] = entry["fetch_bytes"] + entry["write_bytes"]
            roofline["traffic_unit"] = "bytes per launch"
    except (OSError, KeyError, ValueError):
        pass

    # The headline schedule folds every pool, upsample, concat, pad and crop into a convolution, so it has no
    # bandwidth-only dispatch to report.  The stand-alone bandwidth kernels are timed here in a second, unfused
    # schedule of the same network (not part of `value`): hipEvent pairs per dispatch, bytes as each dispatch declares them.
    non_conv = None
    if net == "oidn_unet" and not args.no_unfused_pass:
        ublob = dx.compile_model(model, assume={"H": H, "W": W}, features=networks.UNFUSED_FEATURES, input_layout=lay, output_layout=lay)
        uinst = dx.Module.load(ublob).instance(H=H, W=W)
        uinst.infer_device(ins, None)
        uinst.synchronize()
        uacc = None
        for _ in range(passes):
            t = uinst.bench(warmup=2)
            if uacc is None:
                uacc = t
            else:
                for a2, b2 in zip(uacc, t):
                    a2["latency_ms"] += b2["latency_ms"]
        bw = [a2 for a2 in uacc if not (a2["flops"] > 0 and "conv" in a2["name"])]
        bw_ms = sum(a2["latency_ms"] for a2 in bw) / passes
        bw_bytes = sum(a2["memory_reads"] + a2["memory_writes"] for a2 in bw)
        non_conv = {"dispatches": len(bw), "bytes": bw_bytes, "ms": bw_ms, "GBps": bw_bytes / bw_ms * 1e-6, "frac_of_hbm": bw_bytes / bw_ms * 1e-6 / PEAK_HBM_GBPS,
                    "per_dispatch": [{"name": a2["name"], "in": a2["input"], "out": a2["output"], "GBps": round((a2["memory_reads"] + a2["memory_writes"]) / (a2["latency_ms"] / passes) * 1e-6, 1)} for a2 in bw],
                    "note": "pool / upsample / concat / pad / slice dispatches of the same network compiled with those fusions switched off"}
        del uinst
        if other_ms == 0:
            roofline["non_conv_GBps"] = non_conv["GBps"]
            roofline["non_conv_frac_of_hbm"] = non_conv["frac_of_hbm"]
            roofline["non_conv_source"] = "unfused second schedule (the timed schedule has no bandwidth-only dispatch)"

    # (the library launches lists of up to four dispatches one by one, and any list under DENOX_HIP_NO_GRAPH)
    launched = "in one hipGraph" if mod.runtime_model.dispatch_count > 4 and "DENOX_HIP_NO_GRAPH" not in os.environ else "as plain launches"
    line = {
        "metric": "oidn_unet_fp16_hwc_1080p_throughput" if workload == "oidn_1080p" else f"{workload}_throughput", "value": H * W / (ms * 1e-3) * 1e-6, "unit": "Mpix/s",
        "n_gpus": 1, "steps": steps, "warmup": warmup, "ms_per_step": ms, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "f16", "data": "synthetic",
        "config": {"workload": f"{description}; {mod.runtime_model.dispatch_count} dispatches {launched}", "device_bytes": inst.device_bytes,
                   "schedule": "min-cost over measured dispatch latencies" if db is not None else "min-cost over roofline estimates",
                   "tuning_seconds": round(tune_s, 2), "host_pointer_path_ms_per_frame": round(host_ms, 3), "host_pointer_pipelined_ms_per_frame": round(pipelined_ms, 3),
                   "two_frames_in_flight_ms_per_frame": round(two_ms, 4) if two_ms else None,
                   "two_frames_in_flight_Mpix_s": round(H * W / (two_ms * 1e-3) * 1e-6, 1) if two_ms else None,
                   "single_replay_ms_median": round(singles[len(singles) // 2], 4), "single_replay_ms_p95": round(singles[int(len(singles) * 0.95)], 4),
                   "settle_seconds": args.settle_seconds,
                   "layout_preference": args.layout_preference, "internal_tensors_in_chwc8": chwc8, "schedule_configs": chosen,
                   "schedule_kernels": [d["entry_point"] for d in desc]},
        "roofline": roofline,
    }
    if non_conv is not None:
        line["non_conv_kernels"] = non_conv
    rc = 0
    if not args.no_cpu_baseline:
        line["cpu_baseline"] = cpu_baseline(net, net_kw, args.seed, H, W, out_hwc)
        line["parity"] = line["cpu_baseline"]["parity"]
        if not line["parity"]["ok"]:
            print(f"bench.py: the timed schedule's output misses the parity bar: {line['parity']}", file=sys.stderr)
            rc = 1
    return line, rc


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--workload", default="oidn_1080p", choices=sorted(WORKLOADS),
                    help="oidn_1080p is the headline configuration; the others are the remaining benchmark configurations")
    ap.add_argument("--height", type=int, default=None)
    ap.add_argument("--width", type=int, default=None)
    ap.add_argument("--seed", type=int, default=0)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--per-dispatch", action="store_true", help="print the per-dispatch report to stderr")
    ap.add_argument("--conv-config", default=None)
    ap.add_argument("--db", default=None, help="timing table to select the schedule with (default: measure one now)")
    ap.add_argument("--no-tune", action="store_true", help="skip the timing table; select by roofline estimates")
    ap.add_argument("--layout-preference", type=int, default=0,
                    help="1: candidates that read or write a channel-block-major (CHWC8) internal tensor count half their cost, which "
                         "forces that layout wherever it exists; 0 (default): the measured cost alone decides")
    ap.add_argument("--no-upsample-fold", action="store_true", help="no kernels that fold a fused 2x upsample into the weights")
    ap.add_argument("--no-blocked-layout", action="store_true", help="internal tensors pixel-major (HWC) only: no CHWC8 candidates")
    ap.add_argument("--no-unfused-pass", action="store_true", help="skip the second, unfused schedule that times the stand-alone bandwidth kernels")
    ap.add_argument("--settle-seconds", type=float, default=0.3, help="untimed back-to-back frames before --warmup, until clocks have settled")
    ap.add_argument("--no-two-frames", action="store_true",
                    help="skip the two-frames-in-flight figure (under a profiler its overlapping kernels would blur the per-kernel durations)")
    ap.add_argument("--no-other-workloads", action="store_true",
                    help="only the selected workload; by default the headline run appends short runs of the other benchmark configurations")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py: this path runs on exactly one GPU (independent frames shard trivially across GPUs; "
              "nothing in this build uses a second one). Run with --gpus 1.", file=sys.stderr)
        return 2

    import torch
    if not torch.cuda.is_available():
        print("bench.py: no GPU visible", file=sys.stderr)
        return 1
    line, rc = measure(args, args.workload, args.steps, args.warmup, brief=False)
    if line is None:
        return rc
    # The other benchmark configurations (parity-test cases, not the headline), each tuned, timed briefly and checked on oracle
    # crops after the headline's timed region; they never enter `value`.
    if args.workload == "oidn_1080p" and not args.no_other_workloads and args.height is None and args.width is None:
        others = []
        t0 = time.perf_counter()
        for w in OTHER_WORKLOADS:
            o, orc = measure(args, w, OTHER_STEPS, OTHER_WARMUP, brief=True)
            if o is None:
                o = {"workload": w, "error": "non-finite output"}
            elif orc:
                print(f"bench.py: {w}: the timed schedule's output misses the parity bar: {o['parity']}", file=sys.stderr)
            rc = rc or orc
            others.append(o)
        line["other_workloads"] = others
        line["other_workloads_seconds"] = round(time.perf_counter() - t0, 1)
    print(json.dumps(line))
    return rc


if __name__ == "__main__":
    sys.exit(main())
