"""Planar (CHW) interfaces of tensors with whole 8-channel groups: the tiled transpose of relayout.hip in both directions, bit for
bit against numpy.  Channel counts on both sides of its tile sizes (32, 64, 128, 256 channels) and group counts that are no powers of
two; extents whose pixel count is below one block, a multiple of the tile, and neither (planes then start at odd addresses)."""
import numpy as np
import pytest

import denox_amd as dx
from util import assert_bits_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C", [8, 16, 24, 32, 40, 64, 72, 96, 128, 136, 256, 264])
@pytest.mark.parametrize("H,W", [(1, 1), (1, 7), (3, 5), (16, 64), (37, 71), (64, 80)])
def test_planar_interface(C, H, W):
    rng = np.random.default_rng(C + H * W)
    m = dx.Model()
    m.output(m.relu(m.input("x", "W", "H", C)), "y")
    x = rng.standard_normal((H, W, C)).astype(np.float16)
    want = np.where(x > 0, x, np.float16(0))  # (the layer gives +0 for -0, np.maximum need not)
    planar = np.ascontiguousarray(x.transpose(2, 0, 1))
    got = dx.Module.compile(m, input_layout=dx.Layout.CHW).instance(H=H, W=W).infer(planar)[0]
    assert_bits_equal(got, want, f"CHW -> HWC {C} {H}x{W}")
    got = dx.Module.compile(m, output_layout=dx.Layout.CHW).instance(H=H, W=W).infer(x)[0]
    assert_bits_equal(got, np.ascontiguousarray(want.transpose(2, 0, 1)), f"HWC -> CHW {C} {H}x{W}")
