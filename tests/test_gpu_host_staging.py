"""The blocking call on large pageable arrays (host_staging.cpp: a ring of four page-locked chunks of 4 MiB): copies only, so
the result has the bits of the same call through small or page-locked arrays.  Sizes around the 4 MiB threshold, one chunk more and
less, several inputs and outputs, arrays larger than the ring, and calls from two threads on two instances."""
import threading

import numpy as np
import pytest

import denox_amd as dx
from util import assert_bits_equal

pytestmark = pytest.mark.gpu


def module(C):
    m = dx.Model()
    a, b = m.input("a", "W", "H", C), m.input("b", "W", "H", C)
    m.output(m.relu(a), "r")
    m.output(m.concat(b, a), "c")
    return dx.Module.compile(m)


def data(rng, H, W, C):
    return [rng.integers(0, 0x7C00, (H, W, C), dtype=np.uint16).view(np.float16) for _ in range(2)]


def check(inst, a, b):
    r, c = inst.infer(a, b)
    assert_bits_equal(r, a, "relu of non-negative values")
    assert_bits_equal(c, np.concatenate([b, a], axis=2), "concat")


# bytes of one input: 8 * 2 * H * W
@pytest.mark.parametrize("H,W", [(512, 511), (512, 512), (512, 513), (769, 512), (1023, 1025), (2100, 2500)])
def test_pageable_arrays(H, W):
    rng = np.random.default_rng(H + W)
    inst = module(8).instance(H=H, W=W)
    for _ in range(2):
        check(inst, *data(rng, H, W, 8))


def test_page_locked_and_pageable_mixed():
    rng = np.random.default_rng(3)
    inst = module(8).instance(H=700, W=701)
    a, b = data(rng, 700, 701, 8)
    pinned = dx.pinned_empty(a.shape)
    pinned[...] = a
    check(inst, pinned, b)
    check(inst, a, pinned)


def test_two_threads():
    mod = module(8)
    insts = [mod.instance(H=640, W=640), mod.instance(H=641, W=600)]
    errors = []

    def work(inst, H, W, seed):
        try:
            rng = np.random.default_rng(seed)
            for _ in range(3):
                check(inst, *data(rng, H, W, 8))
        except Exception as e:  # noqa: BLE001 -- reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(insts[0], 640, 640, 1)), threading.Thread(target=work, args=(insts[1], 641, 600, 2))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
