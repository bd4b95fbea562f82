"""Convolutions whose weights and halos go straight into LDS (conv3x3_mfma_dl.hip) at the edges of what they do: one pixel, one tile and a
pixel more or less (tiles of 32 columns and 16 or 32 rows), several units per workgroup, one step and many, slices of 32 to 128 output
channels and channels past the last one, a pooled result of odd extents, a result inside a concat, both layouts of source and result.

Inputs, weights and bias are small integers: every product and partial sum is exact in binary32 (at most 9 * 256 * 2 + 3 < 2^24) and every
result within 2048 in magnitude is exact in binary16, so the result has the oracle's bits whatever the order of the sums."""
import numpy as np
import pytest

import denox_amd as dx
from util import assert_bits_equal, integer_conv_on_gpu

pytestmark = pytest.mark.gpu

# C, K, H, W, pooled
SHAPES = [(16, 32, 1, 1, False), (16, 8, 2, 3, True), (32, 64, 16, 32, False), (32, 48, 33, 65, True), (64, 64, 31, 31, False), (64, 96, 34, 66, True), (96, 128, 17, 97, False),
          (128, 160, 20, 40, True), (112, 112, 65, 33, False), (192, 192, 15, 70, False), (256, 64, 9, 130, False), (64, 64, 300, 420, False), (32, 96, 270, 510, True)]

CONFIGS = ["l8k32", "l8k16"]  # 32 and 16 channels per step


def blocked(x):
    H, W, C = x.shape
    return np.ascontiguousarray(x.reshape(H, W, C // 8, 8).transpose(2, 0, 1, 3))


def planar(y):
    g, H, W, _ = y.shape
    return y.transpose(1, 2, 0, 3).reshape(H, W, g * 8)


SOURCE = "conv3x3_mfma_dl.hip"


@pytest.mark.parametrize("config", CONFIGS)
@pytest.mark.parametrize("C,K,H,W,pooled", SHAPES)
def test_streamed_into_lds_equals_the_definition(oracle, config, C, K, H, W, pooled):
    rng = np.random.default_rng(C + K + H)
    m = dx.Model()
    t = m.conv2d(m.input("x", "W", "H", C), rng.choice([-1, 0, 0, 0, 1], (K, C, 3, 3)).astype(np.float16), rng.integers(-3, 4, K).astype(np.float16))
    t = m.activation(t, "leaky_relu", 0.5) if K % 64 else m.relu(t)
    if pooled:
        t = m.pool(t)
    m.output(t, "out")
    x = rng.integers(-2, 3, (H, W, C)).astype(np.float16)
    want = oracle.run_graph(m.to_ops({"H": H, "W": W}), {"x": x}, "fp32")[t.name]
    assert np.abs(want).max(initial=0) < 1024  # (a leaky slope of 1/2 leaves at most one bit below 1)
    for blocked_in in (False, True):
        for blocked_out in (False, True):
            layouts = dict(input_layout=dx.Layout.CHWC8 if blocked_in else dx.Layout.HWC, output_layout=dx.Layout.CHWC8 if blocked_out else dx.Layout.HWC)
            if C % int(config[-2:]):  # whole steps of channels only
                with pytest.raises(dx.DenoxHipError) as e:
                    dx.compile_model(m, conv_config=config, assume={"H": H, "W": W}, **layouts)
                assert e.value.status == 5
                continue
            blob = dx.compile_model(m, conv_config=config, assume={"H": H, "W": W}, **layouts)
            assert [d["src_path"] for d in dx.describe(blob, H=H, W=W)["dispatches"]] == [SOURCE]
            got = dx.Module.load(blob).instance(H=H, W=W).infer(blocked(x) if blocked_in else x)[0]
            assert_bits_equal(planar(got) if blocked_out else got, want.astype(np.float16), f"{config} {layouts}")


# filter, stride, padding (y, x), C, K, H, W: phases of unequal taps, padding past the image, extents that leave a phase a row or column short
STRIDED = [((5, 5), (2, 2), (2, 2), 32, 64, 45, 131), ((5, 5), (1, 1), (2, 2), 16, 40, 20, 70), ((4, 4), (2, 2), (1, 1), 32, 32, 34, 66), ((7, 3), (2, 1), (3, 0), 16, 64, 41, 37),
           ((3, 7), (1, 2), (5, 2), 32, 96, 18, 140), ((2, 2), (1, 1), (0, 0), 48, 128, 33, 33), ((5, 5), (2, 2), (0, 4), 64, 48, 5, 40)]


@pytest.mark.parametrize("config", CONFIGS)
@pytest.mark.parametrize("filt,stride,pad,C,K,H,W", STRIDED)
def test_strides_and_filters(oracle, config, filt, stride, pad, C, K, H, W):
    rng = np.random.default_rng(sum(filt) + C + K)
    m = dx.Model()
    t = m.relu(m.conv2d(m.input("x", "W", "H", C), rng.choice([-1, 0, 0, 0, 1], (K, C) + filt).astype(np.float16), rng.integers(-3, 4, K).astype(np.float16), stride=stride, padding=pad))
    m.output(t, "out")
    x = rng.integers(-2, 3, (H, W, C)).astype(np.float16)
    want = oracle.run_graph(m.to_ops({"H": H, "W": W}), {"x": x}, "fp32")[t.name]
    assert np.abs(want).max(initial=0) < 2048
    for blocked_in in (False, True):
        layout = dx.Layout.CHWC8 if blocked_in else dx.Layout.HWC
        if C % int(config[-2:]):  # whole steps of channels only
            with pytest.raises(dx.DenoxHipError) as e:
                dx.compile_model(m, conv_config=config, assume={"H": H, "W": W}, input_layout=layout)
            assert e.value.status == 5
            continue
        blob = dx.compile_model(m, conv_config=config, assume={"H": H, "W": W}, input_layout=layout)
        assert [d["src_path"] for d in dx.describe(blob, H=H, W=W)["dispatches"]] == [SOURCE]
        assert_bits_equal(dx.Module.load(blob).instance(H=H, W=W).infer(blocked(x) if blocked_in else x)[0], want.astype(np.float16), f"{config} {layout}")


# filter, stride, padding, C, K, H, W, pooled, layouts of source and result: two and more units for every workgroup (256 of them), with results kept for
# the next unit's steps (one step, several, several phases) and stored at once (128 channels), several slices, a pooled result
MANY_UNITS = [
    ("l8k32", (3, 3), (1, 1), (1, 1), 64, 64, 544, 960, False, False, False), ("l8k32", (3, 3), (1, 1), (1, 1), 32, 32, 600, 1000, False, False, True),
    ("l8k32", (3, 3), (1, 1), (1, 1), 96, 128, 545, 963, True, True, True), ("l8k16", (3, 3), (1, 1), (1, 1), 64, 64, 1088, 960, False, True, True),
    ("l8k16", (3, 3), (1, 1), (1, 1), 48, 96, 700, 1000, True, False, False), ("l8k16", (3, 3), (1, 1), (1, 1), 128, 160, 270, 480, False, True, False),
    ("l8k32", (5, 5), (2, 2), (2, 2), 32, 64, 1080, 1920, False, False, False), ("l8k16", (5, 5), (2, 2), (2, 2), 48, 128, 1080, 1920, False, True, True),
    ("l8k32", (4, 4), (2, 2), (1, 1), 64, 96, 1001, 1441, False, True, False), ("l8k16", (7, 3), (2, 1), (3, 0), 16, 64, 1203, 901, False, False, True),
    ("l8k16", (7, 7), (1, 1), (3, 3), 32, 64, 270, 520, False, False, False),
]


@pytest.mark.parametrize("config,filt,stride,pad,C,K,H,W,pooled,blocked_in,blocked_out", MANY_UNITS)
def test_many_units_per_workgroup(config, filt, stride, pad, C, K, H, W, pooled, blocked_in, blocked_out):
    """What only a second unit of work reaches: halo offsets moved from the last phase of one unit to the first of the next, stores of a
    finished tile during the next one's steps, the parity of the two LDS buffers.  Twice: the same bits."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(C + H)
    w, b = rng.choice([-1, 0, 0, 0, 1], (K, C) + filt).astype(np.float16), rng.integers(-3, 4, K).astype(np.float16)
    m = dx.Model()
    t = m.relu(m.conv2d(m.input("x", "W", "H", C), w, b, stride=stride, padding=pad))
    m.output(m.pool(t) if pooled else t, "out")
    blob = dx.compile_model(m, conv_config=config, assume={"H": H, "W": W}, input_layout=dx.Layout.CHWC8 if blocked_in else dx.Layout.HWC,
                            output_layout=dx.Layout.CHWC8 if blocked_out else dx.Layout.HWC)
    d, = dx.describe(blob, H=H, W=W)["dispatches"]
    info = dict(kv.split("=") for kv in d["debug_info"].split(" | ")[1].split())
    x = rng.integers(-2, 3, (H, W, C)).astype(np.float16)
    want = torch.relu(integer_conv_on_gpu(x, w, b, stride, pad))
    oh, ow = want.shape[:2]
    assert d["src_path"] == SOURCE and -(-ow // 32) * -(-oh // (8 * int(info["RPW"]))) * (-(-K // 32) * 32 // int(info["KT"])) >= 2 * d["workgroup_count"][0]
    assert float(want.max()) < 2048
    if pooled:
        want = want[:oh // 2 * 2, :ow // 2 * 2].reshape(oh // 2, 2, ow // 2, 2, K).amax((1, 3))
    want = want.half().cpu().numpy()
    inst = dx.Module.load(blob).instance(H=H, W=W)
    for _ in range(2):
        got = inst.infer(blocked(x) if blocked_in else x)[0]
        assert_bits_equal(planar(got) if blocked_out else got, want, config)


def test_result_inside_a_concat(oracle):
    """The concat's sources written in place: a pixel pitch of two tensors, 16-byte aligned at the second one's first channel."""
    rng = np.random.default_rng(5)
    H, W = 35, 68
    m = dx.Model()
    x = m.input("x", "W", "H", 32)
    conv = lambda k: m.relu(m.conv2d(x, rng.choice([-1, 0, 0, 1], (k, 32, 3, 3)).astype(np.float16), rng.integers(-3, 4, k).astype(np.float16)))  # noqa: E731
    t = m.concat(conv(64), conv(40))
    m.output(t, "out")
    v = rng.integers(-2, 3, (H, W, 32)).astype(np.float16)
    want = oracle.run_graph(m.to_ops({"H": H, "W": W}), {"x": v}, "fp32")[t.name]
    for config in CONFIGS:
        blob = dx.compile_model(m, conv_config=config, assume={"H": H, "W": W})
        assert [d["src_path"] for d in dx.describe(blob, H=H, W=W)["dispatches"]] == [SOURCE] * 2
        assert_bits_equal(dx.Module.load(blob).instance(H=H, W=W).infer(v)[0], want.astype(np.float16), config)
