"""Convolutions over an upsampled source with the products of a low-resolution pixel shared between its outputs (conv3x3_upshare.hip), at the
edges of its tiles: strips of 31 source pixels, 8 or 16 output rows per workgroup, 62 stored columns, steps of 16 and 32 channels,
partial vectors of the second source, slices and blocks of output channels past the last one, both layouts of every tensor.

Inputs, weights and bias are small integers: every product and every partial sum is exact in binary32 (at most 9 * 224 * 2 * 2 + 3 < 2^24)
and every result within 2048 in magnitude is exact in binary16, so the result has the oracle's bits whatever the order of the sums."""
import numpy as np
import pytest

import denox_amd as dx
from util import assert_bits_equal, integer_conv_on_gpu

pytestmark = pytest.mark.gpu

# CA (upsampled), CB, K, H, W of the result, replicate-padded second source.  Steps of 32 channels of A where they are whole, else of 16.
ONE_ROW = [  # slices of 32 channels beside a second source: two rows of them do not fit the LDS
    (8, 8, 8, 2, 2, False), (16, 16, 32, 16, 62, False), (48, 12, 96, 62, 66, True), (112, 48, 96, 66, 130, False), (32, 64, 224, 14, 18, False),
]
BOTH = [
    (64, 9, 64, 34, 124, True), (64, 0, 64, 32, 126, False), (32, 24, 40, 18, 64, False), (24, 73, 48, 30, 60, True), (96, 32, 128, 4, 250, False),
    (224, 20, 64, 10, 38, False), (64, 9, 128, 130, 310, True), (48, 12, 64, 36, 72, True), (64, 16, 64, 34, 126, True), (32, 0, 96, 34, 64, False),
    # steps of 16 channels: block-major sources, no second source, a last group of 8 channels of A, the second source through registers
    (48, 16, 64, 34, 66, False), (112, 48, 128, 18, 126, False), (48, 0, 40, 36, 62, False), (16, 0, 64, 2, 64, False), (24, 73, 64, 20, 68, True), (80, 73, 64, 34, 70, False),
    (96, 32, 112, 4, 250, False),
]
SHAPES = BOTH + ONE_ROW
CONFIGS = ["e8r2", "e8r1"]  # two rows per wave and one


def blocked(x):
    H, W, C = x.shape
    return np.ascontiguousarray(x.reshape(H, W, C // 8, 8).transpose(2, 0, 1, 3))


def planar(y):
    g, H, W, _ = y.shape
    return y.transpose(1, 2, 0, 3).reshape(H, W, g * 8)


def layer(CA, CB, K, H, W, padded, rng, act="relu"):
    m = dx.Model()
    feeds = {"lo": rng.integers(-2, 3, (H // 2, W // 2, CA)).astype(np.float16)}
    t = m.upsample(m.input("lo", m.sym("W") // 2, m.sym("H") // 2, CA))
    if CB:
        h, w = (H - 3, W - 5) if padded else (H, W)
        feeds["x"] = rng.integers(-2, 3, (h, w, CB)).astype(np.float16)
        x = m.input("x", m.sym("W") - 5, m.sym("H") - 3, CB) if padded else m.input("x", "W", "H", CB)
        t = m.concat(t, m.pad(x, 2, 3, 1, 2) if padded else x)
    w = rng.choice([-1, 0, 0, 0, 1], (K, CA + CB, 3, 3)).astype(np.float16)
    t = m.conv2d(t, w, rng.integers(-3, 4, K).astype(np.float16))
    if act != "none":
        t = m.activation(t, act, 0.5)
    m.output(t, "out")
    return m, t, feeds


@pytest.mark.parametrize("config,CA,CB,K,H,W,padded", [("e8r2",) + s for s in BOTH] + [("e8r1",) + s for s in SHAPES])
def test_shared_products_equal_the_definition(oracle, config, CA, CB, K, H, W, padded):
    rng = np.random.default_rng(CA + CB + K)
    m, t, feeds = layer(CA, CB, K, H, W, padded, rng, "leaky_relu" if K % 64 else "relu")
    want = oracle.run_graph(m.to_ops({"H": H, "W": W}), feeds, "fp32")[t.name]
    assert np.abs(want).max() < 2048  # (a leaky slope of 1/2 leaves at most one bit below 1)
    for blocked_in in (False, True):
        for blocked_out in (False, True):
            if blocked_in and (CA % 16 or CB % 8):
                continue  # whole steps and vectors only
            layouts = dict(input_layout=dx.Layout.CHWC8 if blocked_in else dx.Layout.HWC, output_layout=dx.Layout.CHWC8 if blocked_out else dx.Layout.HWC)
            blob = dx.compile_model(m, conv_config=config, assume={"H": H, "W": W}, **layouts)
            d = dx.describe(blob, H=H, W=W)["dispatches"]
            assert [x["src_path"] for x in d] == ["conv3x3_upshare.hip"]
            xs = [feeds[k] for k in ("lo", "x") if k in feeds]
            got = dx.Module.load(blob).instance(H=H, W=W).infer(*[blocked(x) if blocked_in else x for x in xs])[0]
            assert_bits_equal(planar(got) if blocked_out else got, want.astype(np.float16), f"{config} {layouts}")


# CA, CB, K, H, W, padded, layouts of sources and result: two and more units for every workgroup (256 of them), among them units inside the image one
# after the other, the last ones of an XCD, a result above 192 MiB (stored past the cache) and units of several slices
MANY_UNITS = [
    ("e8r2", 64, 9, 64, 1088, 1920, True, False, False), ("e8r2", 64, 16, 64, 1088, 1920, False, True, True), ("e8r2", 48, 16, 64, 500, 1000, False, True, False),
    ("e8r2", 64, 0, 64, 500, 1002, False, False, True), ("e8r2", 128, 9, 128, 300, 960, True, False, False), ("e8r2", 32, 24, 64, 542, 960, False, False, True),
    ("e8r1", 64, 9, 64, 542, 960, True, False, False), ("e8r1", 96, 32, 64, 400, 1000, False, True, True), ("e8r1", 112, 48, 96, 400, 480, False, False, True),
]


@pytest.mark.parametrize("config,CA,CB,K,H,W,padded,blocked_in,blocked_out", MANY_UNITS)
def test_many_units_per_workgroup(config, CA, CB, K, H, W, padded, blocked_in, blocked_out):
    """What only a second unit of work reaches: halo offsets moved from one unit to the next, its first step loaded while the last one's result
    is on its way out, the parity of the two LDS buffers.  Twice: the same bits."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(CA + H)
    m, t, feeds = layer(CA, CB, K, H, W, padded, rng)
    blob = dx.compile_model(m, conv_config=config, assume={"H": H, "W": W}, input_layout=dx.Layout.CHWC8 if blocked_in else dx.Layout.HWC,
                            output_layout=dx.Layout.CHWC8 if blocked_out else dx.Layout.HWC)
    d, = dx.describe(blob, H=H, W=W)["dispatches"]
    info = dict(kv.split("=") for kv in d["debug_info"].split(" | ")[1].split())
    rows = 2 * (8 // (int(info["KT"]) // 32)) * int(info["RPW"])
    assert d["src_path"] == "conv3x3_upshare.hip" and -(-W // 62) * -(-(H + 1) // rows) * (-(-K // 32) * 32 // int(info["KT"])) >= 2 * d["workgroup_count"][0]
    x = np.zeros((H, W, CA + CB), np.float16)
    x[:, :, :CA] = feeds["lo"].repeat(2, 0).repeat(2, 1)
    if CB:
        x[:, :, CA:] = np.pad(feeds["x"], ((1, 2), (2, 3), (0, 0)), "edge") if padded else feeds["x"]
    conv, = [op for op in m.to_ops({"H": H, "W": W}) if "weight" in op]
    want = torch.relu(integer_conv_on_gpu(x, conv["weight"], conv["bias"]))
    assert float(want.max()) < 2048
    want = want.half().cpu().numpy()
    inst = dx.Module.load(blob).instance(H=H, W=W)
    xs = [feeds[k] for k in ("lo", "x") if k in feeds]
    for _ in range(2):
        got = inst.infer(*[blocked(v) if blocked_in else v for v in xs])[0]
        assert_bits_equal(planar(got) if blocked_out else got, want, config)


@pytest.mark.parametrize("config", CONFIGS)
def test_not_a_number_reaches_its_neighbours_only(config):
    """An infinity and a NaN of either source: exactly the outputs whose taps cover them are affected (padding channels, lanes that only
    supply an edge and positions outside the image multiply zeros, never what memory holds there)."""
    rng = np.random.default_rng(3)
    H, W = 36, 130
    m, t, feeds = layer(64, 9, 64, H, W, False, rng, "none")
    feeds["lo"][7, 31, 5] = np.inf
    feeds["x"][20, 62, 8] = np.nan
    blob = dx.compile_model(m, conv_config=config, assume={"H": H, "W": W})
    assert dx.describe(blob, H=H, W=W)["dispatches"][0]["src_path"] == "conv3x3_upshare.hip"
    got = dx.Module.load(blob).instance(H=H, W=W).infer(feeds["lo"], feeds["x"])[0]
    bad = ~np.isfinite(got.astype(np.float32)).all(axis=2)
    want = np.zeros((H, W), bool)
    want[13:17, 61:65] = True  # source pixel (7, 31) is outputs 14 - 15 x 62 - 63, and one more on each side
    want[19:22, 61:64] = True
    assert (bad == want).all(), np.argwhere(bad != want)[:8]


@pytest.mark.parametrize("config", CONFIGS)
@pytest.mark.parametrize("blocked_out", [False, True])
def test_rows_outside_the_image_are_not_written(config, blocked_out):
    """Every first tile computes the row in front of the image and most last tiles rows behind it: with the result in the middle of a
    larger buffer, nothing around it changes."""
    torch = pytest.importorskip("torch")
    H, W, K = 38, 70, 64
    m, t, feeds = layer(64, 9, K, H, W, False, np.random.default_rng(4))
    blob = dx.compile_model(m, conv_config=config, assume={"H": H, "W": W}, output_layout=dx.Layout.CHWC8 if blocked_out else dx.Layout.HWC)
    assert dx.describe(blob, H=H, W=W)["dispatches"][0]["src_path"] == "conv3x3_upshare.hip"
    inst = dx.Module.load(blob).instance(H=H, W=W)
    want = inst.infer(feeds["lo"], feeds["x"])[0].reshape(-1).view(np.int16)
    size, margin = H * W * K, 40 * W * K  # (more than the tiles' rows past the image, as planes or as whole pixels)
    buf = torch.full((size + 2 * margin,), 0x5A5A, dtype=torch.int16, device="cuda")
    d_in = [torch.from_numpy(feeds[k]).cuda() for k in ("lo", "x")]
    torch.cuda.synchronize()
    inst.infer_device([d.data_ptr() for d in d_in], [buf.data_ptr() + 2 * margin])
    inst.synchronize()
    got = buf.cpu().numpy()
    assert (got[:margin] == 0x5A5A).all() and (got[margin + size:] == 0x5A5A).all()
    np.testing.assert_array_equal(got[margin:margin + size], want)
