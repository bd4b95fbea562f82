"""Interface tensors that the caller keeps in CHWC8 and that kernels read and write in that layout, against the same model with an
HWC interface: bit for bit (the same convolution configuration, copies and element-wise operations elsewhere).  Models in which such
a tensor meets what needs memory of its own: a concat of two inputs (no aliasing of caller memory), an input with several
readers, one of which takes HWC only, an output that is read again, a tensor that is input and output of nothing else."""
import numpy as np
import pytest

import denox_amd as dx
from util import assert_bits_equal, he_weights, small_bias

pytestmark = pytest.mark.gpu


def blocked(x):
    H, W, C = x.shape
    return np.ascontiguousarray(x.reshape(H, W, C // 8, 8).transpose(2, 0, 1, 3))


def planar(y):
    g, H, W, _ = y.shape
    return y.transpose(1, 2, 0, 3).reshape(H, W, g * 8)


def conv(m, rng, t, K):
    return m.conv2d(t, he_weights(rng, K, t.channels), small_bias(rng, K))


def build(kind, m, rng, C):
    x = m.input("x", "W", "H", C)
    if kind == "conv":
        return [conv(m, rng, x, 32)]
    if kind == "pool_upsample":
        return [m.upsample(m.pool(x)), m.relu(x)]
    if kind == "concat_of_inputs":
        return [m.concat(x, m.input("y", "W", "H", C))]
    if kind == "two_readers":
        return [m.relu(conv(m, rng, x, 16)), m.slice(x, 1, "W", 0, "H")]
    if kind == "output_read_again":
        y = m.relu(conv(m, rng, x, 16))
        return [y, conv(m, rng, y, 8)]
    raise KeyError(kind)


@pytest.mark.parametrize("kind", ["conv", "pool_upsample", "concat_of_inputs", "two_readers", "output_read_again"])
@pytest.mark.parametrize("C,H,W", [(8, 4, 6), (24, 38, 70)])
@pytest.mark.parametrize("layouts", [("CHWC8", "CHWC8"), ("CHWC8", "HWC"), ("HWC", "CHWC8")])
def test_blocked_interface_equals_hwc(kind, C, H, W, layouts):
    rng = np.random.default_rng(C + H)
    m = dx.Model()
    outs = build(kind, m, rng, C)
    for i, t in enumerate(outs):
        m.output(t, f"o{i}")
    xs = [rng.standard_normal((H, W, C)).astype(np.float16) for _ in m.inputs]
    want = dx.Module.compile(m, conv_config="s8r2k16").instance(H=H, W=W).infer(*xs)
    li, lo = (dx.Layout[n] for n in layouts)
    inst = dx.Module.compile(m, conv_config="s8r2k16", input_layout=li, output_layout=lo).instance(H=H, W=W)
    got = inst.infer(*[blocked(x) if layouts[0] == "CHWC8" else x for x in xs])
    for i, (g, w) in enumerate(zip(got, want)):
        assert_bits_equal(planar(g) if layouts[1] == "CHWC8" else g, w, f"{kind} output {i}")


def test_conv_between_blocked_interfaces_is_one_dispatch():
    rng = np.random.default_rng(1)
    m = dx.Model()
    m.output(conv(m, rng, m.input("x", "W", "H", 64), 64), "o0")
    both = dict(input_layout=dx.Layout.CHWC8, output_layout=dx.Layout.CHWC8)
    assert dx.Module.compile(m, **both).runtime_model.dispatch_count == 1
    assert dx.Module.compile(m, features=dict(blocked_layout=False), **both).runtime_model.dispatch_count == 3
