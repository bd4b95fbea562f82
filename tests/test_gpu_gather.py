"""Chains of data-movement layers in one dispatch (gather.hip; pool.hip through a pad) against the same layers as dispatches of
their own, bit for bit, and against the oracle: copies and element-wise binary16 operations have one right result.  Extents
sit at the edges of a workgroup's pixel run (PQ = 256 pixels for narrow tensors, fewer for wide ones), channel counts on both sides
of the 16-byte vector, with odd and even pixel sizes (word alignment of the rows); NaNs of several payloads."""
import numpy as np
import pytest

import denox_amd as dx
from util import assert_bits_equal

pytestmark = pytest.mark.gpu

SEPARATE = dict(conv_relu_fusion=False, concat_conv_fusion=False, upsample_fusion=False, pad_fusion=False, slice_fusion=False, implicit_concat=False)


def layers(func):
    def chain(m, x):
        p = m.pad_to_multiple(x, 2)
        y = m.concat(m.upsample(m.pool(p, func=func)), p)
        return m.slice(m.activation(y, "leaky_relu", 0.1), 0, x.width, 0, x.height)
    return chain


CHAINS = {
    "layers_max": (layers("max"), 2), "layers_avg": (layers("avg"), 2),
    "upsample_concat": (lambda m, x: m.relu(m.concat(m.upsample(m.pool(x)), x)), 2),  # needs even extents
    "pad_relu_slice": (lambda m, x: m.slice(m.relu(m.pad(x, 3, 2, 1, 4)), 2, x.width + 4, 1, x.height + 3), 1),
    "pad_pool": (lambda m, x: m.pool(m.pad(x, 3, 5, 2, 7), kernel=(3, 2)), 1),
    "pad_twice": (lambda m, x: (lambda p: m.relu(m.concat(p, p)))(m.pad(x, 1, 0, 2, 1)), 1),
    "upsample3_leaky": (lambda m, x: m.activation(m.upsample(x, 3), "leaky_relu", 0.3), 1),
    "second_upsampled": (lambda m, x: m.slice(m.activation(m.concat(x, m.upsample(m.pool(x))), "leaky_relu", 0.1), 1, x.width, 1, x.height), 2),  # (even extents)
    "both_upsampled": (lambda m, x: (lambda p: m.relu(m.concat(m.upsample(p), m.upsample(m.relu(p)))))(m.pool(x)), 3),  # (even extents)
    "padded_pools_in_place_avg": (lambda m, x: m.concat(m.pool(m.pad(x, 2, 0, 0, 3)), m.pool(m.pad(m.relu(x), 0, 2, 3, 0), func="avg")), 3),  # into channel ranges
    "two_pads": (lambda m, x: m.relu(m.concat(m.pad(x, 4, 0, 0, 3), m.pad(m.relu(x), 0, 4, 3, 0))), 1),
}


EVEN = ("upsample_concat", "second_upsampled", "both_upsampled")


@pytest.mark.parametrize("C", [1, 3, 8, 9, 24, 73])
@pytest.mark.parametrize("H,W", [(6, 2), (4, 256), (5, 259), (34, 510)])
@pytest.mark.parametrize("chain", sorted(CHAINS))
def test_chain_equals_separate_layers(oracle, chain, C, H, W):
    build, dispatches = CHAINS[chain]
    if chain in EVEN:
        H, W = H + H % 2, W + W % 2
    rng = np.random.default_rng(C * 1000 + W)
    x = rng.standard_normal((H, W, C)).astype(np.float16)
    x.reshape(-1)[:: 17] = np.float16(-0.0)
    x[0, 0, 0], x[-1, -1, -1] = np.float16(np.inf), np.float16(-np.inf)
    m = dx.Model()
    t = build(m, m.input("input", "W", "H", C))
    m.output(t, "output")
    fused = dx.Module.compile(m)
    assert fused.runtime_model.dispatch_count <= dispatches + (chain == "two_pads")
    got = fused.instance(H=H, W=W).infer(x)[0]
    want = dx.Module.compile(m, features=SEPARATE).instance(H=H, W=W).infer(x)[0]
    assert_bits_equal(got, want, f"{chain} C={C} {H}x{W}")
    if "avg" not in chain:
        ref = oracle.run_graph(m.to_ops({"H": H, "W": W}), {"input": x}, "f16")[t.name]
        np.testing.assert_array_equal(got, np.asarray(ref, np.float16))


@pytest.mark.parametrize("C", [3, 24])
@pytest.mark.parametrize("chain", sorted(CHAINS))
def test_chain_of_nans_equals_separate_layers(chain, C):
    """At most one NaN per pooling window and channel: which of two operands' payloads an addition keeps is not defined."""
    H, W = 12, 34
    rng = np.random.default_rng(C)
    x = rng.standard_normal((H, W, C)).astype(np.float16)
    bits = x.view(np.uint16)
    bits[::4, ::6] = rng.choice(np.array([0x7E00, 0xFE00, 0x7E35, 0xFFFF], np.uint16), bits[::4, ::6].shape)
    m = dx.Model()
    m.output(CHAINS[chain][0](m, m.input("input", "W", "H", C)), "output")
    got = dx.Module.compile(m).instance(H=H, W=W).infer(x)[0]
    want = dx.Module.compile(m, features=SEPARATE).instance(H=H, W=W).infer(x)[0]
    assert_bits_equal(got, want, f"{chain} C={C}")
