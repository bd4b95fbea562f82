"""A convolution whose result is staged through LDS where a tile is a single reduction step (the staged tile is doubled,
conv3x3_mfma_ws.hip), against the fp32 oracle with the bar of the other convolution tests.  32 and 24 channels are one step of the
configurations with 32-channel steps and two of the others, which keep one staged tile."""
import re

import numpy as np
import pytest

import denox_amd as dx
from util import assert_conv_close, he_weights, small_bias

pytestmark = pytest.mark.gpu


def check(oracle, config, C, K, R, S, stride, H, W, layout_out_pitch=0):
    rng = np.random.default_rng(C * 1000 + K + R * 10 + W)
    x = rng.standard_normal((H, W, C)).astype(np.float16)
    m = dx.Model()
    inp = m.input("input", "W", "H", C)
    t = m.relu(m.conv2d(inp, he_weights(rng, K, C, R, S), small_bias(rng, K), stride=stride, padding=(R // 2, S // 2)))
    if layout_out_pitch:  # the result as a channel range of a wider tensor
        t = m.concat(t, m.relu(m.conv2d(inp, he_weights(rng, layout_out_pitch, C, R, S), small_bias(rng, layout_out_pitch), stride=stride, padding=(R // 2, S // 2))))
    m.output(t)
    # a step of 32 channels is not offered where 16 hold them all; everything else has to compile
    if int(re.search(r"k(\d+)", config).group(1)) > -(-C // 16) * 16:
        with pytest.raises(dx.DenoxHipError):
            dx.Module.compile(m, conv_config=config)
        return
    mod = dx.Module.compile(m, conv_config=config)
    got = mod.instance(H=H, W=W).infer(x)[0]
    want = oracle.run_graph(m.to_ops({"H": H, "W": W}), {"input": x}, "fp32")[t.name]
    assert_conv_close(got, want, f"{config} {C}->{K} {R}x{S} stride {stride} {H}x{W}")


# tiles of 8 x 32 (or 4 x 32) output pixels; 256 workgroups: one tile each, fewer, several with a ragged last one, and (270 x 1300: 1394
# tiles of 8 x 32) five and more, so that both halves of the staged tile are written again
@pytest.mark.parametrize("config", ["r4r2k16", "r4r2k16n", "r8r1k16n", "r4r1k16n", "r4r2k32n", "c4r2k32n", "c4r2k16n", "c4r2k16m"])
@pytest.mark.parametrize("C,K", [(3, 32), (9, 64), (16, 16), (32, 64), (24, 72)])
@pytest.mark.parametrize("H,W", [(1, 1), (8, 32), (9, 65), (133, 700), (270, 1300)])
def test_staged_result_by_steps_per_tile(oracle, config, C, K, H, W):
    check(oracle, config, C, K, 3, 3, (1, 1), H, W)


def test_staged_result_with_one_step_per_tile_inside_a_concat(oracle):
    check(oracle, "r4r2k16n", 9, 64, 3, 3, (1, 1), 21, 70, layout_out_pitch=24)
