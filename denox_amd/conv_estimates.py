"""How far the estimates of csrc/compiler/conv_cost.cpp are from this GPU, and what to change when a kernel has changed.

    python3 -m denox_amd.conv_estimates          measures and prints two tables (a few minutes, most of them hiprtc on a cold cache)
    python3 -m denox_amd.conv_estimates --warm   compiles the kernels that needs, without a GPU

Configurations: every one of `conv_config_names()` on the layers it takes, at three extents, against its estimate.  The ratio is that
of the times beyond the launch, the part that the configuration's entry in `kFactor` multiplies: an entry times its ratio is
the entry that fits this GPU; a new configuration starts from 1.2.  (The constants in front of the factors describe a kernel family;
they were fitted by least squares on the logarithm to tables as `Db.dump_csv` writes them, see conv_cost.cpp.)

Networks: a frame with the schedule the estimates choose against one chosen from a timing table, both without folded weights, which
estimates do not take.
"""
import csv
import io
import multiprocessing
import os
import sys
import tempfile
import time

import numpy as np

import denox_amd as dx
from denox_amd import networks

LAUNCH_MS = 5.56e-3  # kLaunchUs
EXTENTS = [(180, 256), (540, 960), (1080, 1920)]
LAYERS = [(9, 64, 3, 1), (32, 32, 3, 1), (64, 64, 3, 1), (96, 96, 3, 1), (128, 48, 3, 1), (32, 64, 5, 2)]  # C, K, filter, stride
FOLDED = [(64, 9, 64), (96, 32, 64)]                                                                     # CA (upsampled), CB, K
PAIRS = [(9, 32, 32), (64, 32, 3)]                                                                       # C, K1, K2
NETWORKS = [("oidn_unet", {}, 187, 251), ("oidn_unet", {}, 720, 1280), ("oidn_unet", {}, 1080, 1920), ("oidn_unet", {"width_mult": 2}, 1077, 1917), ("tiny_unet", {}, 540, 960)]


def _weights(rng, K, C, R=3):
    return (rng.standard_normal((K, C, R, R)) * np.sqrt(2.0 / (R * R * C))).astype(np.float16)


def _models(config):
    rng = np.random.default_rng(0)
    bias = lambda k: np.zeros(k, np.float16)  # noqa: E731
    for C, K, R, s in LAYERS:
        m = dx.Model()
        m.output(m.relu(m.conv2d(m.input("x", "W", "H", C), _weights(rng, K, C, R), bias(K), stride=(s, s), padding=(R // 2, R // 2))))
        yield f"{C}->{K} {R}x{R}/{s}", m, dict(conv_conv_fusion=False)
    for CA, CB, K in FOLDED:
        m = dx.Model()
        t = m.concat(m.upsample(m.input("a", m.sym("W") // 2, m.sym("H") // 2, CA)), m.input("b", "W", "H", CB))
        m.output(m.relu(m.conv2d(t, _weights(rng, K, CA + CB), bias(K))))
        yield f"{CA}up+{CB}->{K}", m, dict(conv_conv_fusion=False)
    for C, K1, K2 in PAIRS:
        m = dx.Model()
        m.output(m.conv2d(m.relu(m.conv2d(m.input("x", "W", "H", C), _weights(rng, K1, C), bias(K1))), _weights(rng, K2, K1), bias(K2)))
        yield f"{C}->{K1}->{K2}", m, {}


def _scheduled(config):
    """(operation, estimated ms) of the last compilation if it is one dispatch in this configuration."""
    lines = [line.split() for line in dx.last_compile_report().splitlines()[1:] if line.strip()]
    return (lines[0][2], float(lines[0][-2])) if len(lines) == 1 and lines[0][1].split("/")[0] == config else None


def _candidates(config):
    """The layers that have a kernel in this configuration, each with its compile options."""
    for name, m, features in _models(config):
        try:
            dx.compile_model(m, conv_config=config, features=features)
        except dx.DenoxHipError:
            continue
        if _scheduled(config) is not None:
            yield name, m, dict(conv_config=config, features=features)


def _warm(config):
    return len(list(_candidates(config)))


def _measure(config):
    rows = []
    for name, m, options in _candidates(config):
        for H, W in EXTENTS:
            at = dict(options, assume={"H": H, "W": W})
            dx.compile_model(m, **at)
            operation, estimate = _scheduled(config)
            with tempfile.TemporaryDirectory() as tmp:
                db = dx.Db(os.path.join(tmp, "t.db"))
                db.populate(m, compile_kernels=False, **at)
                db.bench(filter="conv3x3_pair" if "->" in name.split("->", 1)[1] else "conv3x3_mfma", min_samples=5, max_relative_error=0.05, max_samples=20, save_progress=False)
                table = [r for r in csv.DictReader(io.StringIO(db.dump_csv())) if r["config"].split("/")[0] == config and r["operation"] == operation and "chwc8" not in r["config"]]
            if len(table) == 1:
                rows.append((name, H, W, estimate, float(table[0]["latency_ms"])))
    return rows


def _frame_us(blob, name, H, W):
    inst = dx.Module.load(blob).instance(H=H, W=W)
    inst.infer(networks.synthetic_input(name, H, W).astype(np.float16))
    best = []
    for _ in range(5):
        t = time.perf_counter()
        for _ in range(50):
            inst.infer_device()
        inst.synchronize()
        best.append((time.perf_counter() - t) / 50 * 1e6)
    return float(np.median(best))


def main():
    names = dx.conv_config_names()
    if "--warm" in sys.argv:
        with multiprocessing.Pool(min(8, os.cpu_count() or 1)) as pool:
            print(sum(pool.imap_unordered(_warm, names)), "kernels")
        return 0
    print("| configuration | layers x extents | measured / estimated beyond the launch: median | lowest | highest |\n|---|---|---|---|---|")
    every = []
    for config in names:
        rows = _measure(config)
        ratios = [(m - LAUNCH_MS) / (e - LAUNCH_MS) for _, _, _, e, m in rows if e > 2 * LAUNCH_MS]  # shorter ones are mostly launch
        every += [m / e for _, _, _, e, m in rows]
        if ratios:
            print(f"| {config} | {len(rows)} | {np.median(ratios):.2f} | {min(ratios):.2f} | {max(ratios):.2f} |", flush=True)
        else:
            print(f"| {config} | {len(rows)} | - | - | - |", flush=True)
    print(f"\nAll {len(every)}: measured over estimated time, median {np.median(every):.3f}, half of them between {np.quantile(every, 0.25):.3f} and {np.quantile(every, 0.75):.3f}.\n")
    print("| network | extent | estimates, us a frame | timing table | ratio |\n|---|---|---|---|---|")
    for name, kw, H, W in NETWORKS:
        m = networks.build(name, **kw)[0]
        at = dict(assume={"H": H, "W": W}, features=dict(upsample_fold=False))
        with tempfile.TemporaryDirectory() as tmp:
            db = dx.Db(os.path.join(tmp, "t.db"))
            db.populate(m, **at)
            db.bench(min_samples=10, max_relative_error=0.03, max_samples=50, save_progress=False)
            tuned = _frame_us(dx.compile_model(m, db=db, **at), name, H, W)
        plain = _frame_us(dx.compile_model(m, **at), name, H, W)
        print(f"| {name}{' x' + str(kw['width_mult']) if kw else ''} | {W} x {H} | {plain:.1f} | {tuned:.1f} | {plain / tuned:.3f} |", flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
