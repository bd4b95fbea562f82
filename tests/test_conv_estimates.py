"""Schedules selected without a timing table: what the estimates may decide and what they leave to a caller's table or to a name."""
import os
import re

import numpy as np
import pytest

import denox_amd as dx
from denox_amd import networks
from util import he_weights

EXTENTS = [("oidn_unet", {}, 1080, 1920), ("oidn_unet", {"width_mult": 2}, 540, 960), ("tiny_unet", {}, 540, 960)]


def configs(report=None):
    """Configuration column of the last compilation's schedule, without the layouts behind it."""
    return [line.split()[1].split("/")[0] for line in (report or dx.last_compile_report()).splitlines()[1:] if line.startswith("conv3x3")]


def folding(names):
    return [n for n in names if n[0] in "fgh"]


@pytest.mark.parametrize("net,kw,H,W", EXTENTS)
def test_estimates_do_not_take_folded_weights(net, kw, H, W):
    """The upsample-folding kernels round sums of weights to binary16: less precise than the layer's own weights.  They are a candidate
    of every table and can be forced by name; without either a schedule keeps the weights as they are."""
    model = networks.build(net, **kw)[0]
    dx.compile_model(model, assume={"H": H, "W": W})
    assert len(configs()) >= 3 and not folding(configs()), configs()


def test_a_table_or_a_name_takes_folded_weights(tmp_path):
    one = dx.Model()
    t = one.concat(one.upsample(one.input("a", one.sym("W") // 2, one.sym("H") // 2, 64)), one.input("b", "W", "H", 9))
    one.output(one.conv2d(t, he_weights(np.random.default_rng(0), 64, 73), np.zeros(64, np.float16)))
    dx.compile_model(one, conv_config="h4r2p")
    assert configs() == ["h4r2p"]
    dx.compile_model(one)
    assert configs() and not folding(configs())
    model = networks.build("oidn_unet")[0]
    at = dict(assume={"H": 64, "W": 64})
    db = dx.Db(str(tmp_path / "t.db"))
    db.populate(model, **at)
    rows = [r.split('","')[2] for r in db.dump_csv().splitlines()[1:]]
    assert any(folding([c.split("/")[0]]) for c in rows)
    dx.compile_model(model, db=db, **at)  # rows without a measurement decide as little as none
    assert not folding(configs())
    for i, c in enumerate(rows):
        db.add_sample(i, 1_000.0 if folding([c.split("/")[0]]) else 10_000.0)
        db.add_sample(i, 1_000.0 if folding([c.split("/")[0]]) else 10_000.0)
    dx.compile_model(model, db=db, **at)
    assert folding(configs())


def single_convs(net, **kw):
    """(configuration, estimated ms) of every single convolution of the schedule that compile_model selects without a table."""
    dx.compile_model(networks.build(net)[0], assume={"H": 1080, "W": 1920}, **kw)
    return [(line.split()[1].split("/")[0], float(line.split()[-2])) for line in dx.last_compile_report().splitlines()[1:] if line.startswith("conv3x3_mfma")]


def test_estimates_per_configuration_whatever_is_fused():
    """Switching the conv -> conv fusion off, or forcing one configuration of that kernel, says nothing about how the single
    convolutions are estimated: the layers between keep the choice (and the time) they have by default."""
    default = single_convs("oidn_unet")
    assert len(set(c for c, _ in default)) >= 4
    off = single_convs("oidn_unet", features=dict(conv_conv_fusion=False))
    assert len(off) == 16 and len(set(c for c, _ in off)) >= 4 and [c for c, _ in off] != ["w4r2k16"] * 16
    inner = lambda s: sum(ms for _, ms in s[-12:])  # noqa: E731
    assert inner(off[2:14]) <= 1.02 * inner(default)  # (the pairs at the ends are two layers each)
    forced = single_convs("oidn_unet", conv_config="x4r2k16")
    assert "x4r2k16" in configs()
    assert len(forced) == 12 and inner(forced) <= 1.02 * inner(default)


@pytest.mark.parametrize("net,H,W,layout,taken", [
    ("tiny_unet", 448, 760, "HWC", []), ("tiny_unet", 540, 960, "HWC", []), ("tiny_unet", 532, 1680, "CHW", []), ("tiny_unet", 720, 1280, "HWC", []),  # 16 -> 32 channels
    ("oidn_unet", 187, 251, "HWC", []), ("oidn_unet", 512, 512, "HWC", ["e8r1"]), ("oidn_unet", 1080, 1920, "HWC", ["e8r1", "e8r2", "l8k16", "l8k32"])])
def test_kernels_that_load_into_lds_are_taken_where_they_pay(net, H, W, layout, taken):
    """A launch starts colder inside a frame than behind itself, which the estimates are fitted to.  Measured frames with and without these
    kernels: the small U-Net is up to 3 % slower with them, the U-Net 1 % slower at 187 x 251 and faster at the larger extents."""
    lay = dx.Layout[layout]
    dx.compile_model(networks.build(net)[0], assume={"H": H, "W": W}, input_layout=lay, output_layout=lay)
    assert sorted({c for c in configs() if c[0] in "el"}) == taken


@pytest.mark.parametrize("config", ["x4r2k16", "x8r2k16", "v4r2k64", "y4r2k32", "d4r2k64"])
@pytest.mark.parametrize("H,W", [(16, 30), (64, 64), (300, 61), (1080, 1920)])
def test_forced_pair_is_taken_on_any_extent(config, H, W):
    rng = np.random.default_rng(0)
    m = dx.Model()
    m.output(m.conv2d(m.relu(m.conv2d(m.input("x", "W", "H", 64), he_weights(rng, 32, 64), np.zeros(32, np.float16))), he_weights(rng, 3, 32), np.zeros(3, np.float16)))
    dx.compile_model(m, conv_config=config, assume={"H": H, "W": W})
    assert configs() == [config]
    assert float(re.search(r"estimated_ms=(\S+)", dx.last_compile_report()).group(1)) > 5e-3  # the estimate itself: a launch at least


@pytest.mark.parametrize("C,K,config", [(16, 32, None), (64, 64, None), (256, 256, None), (512, 512, None), (64, 64, "w4r2k16"), (32, 32, "x4r2k16")])
@pytest.mark.parametrize("assume", [{"W": 1, "H": 1}, {"W": 2, "H": 1}, {"W": 0, "H": 64}, {"W": 100_000, "H": 100_000}])
def test_any_assumed_extent_compiles(C, K, config, assume):
    """The assumption guides an estimate and is no limit of the model: one at which a layer has nothing to compute (a pooled image of one
    row, a filter larger than the image) still compiles, as does one beyond any memory."""
    rng = np.random.default_rng(0)
    m = dx.Model()
    t = m.conv2d(m.relu(m.conv2d(m.pool(m.input("x", "W", "H", C)), he_weights(rng, K, C), np.zeros(K, np.float16))), he_weights(rng, K, K), np.zeros(K, np.float16))
    m.output(m.conv2d(t, he_weights(rng, K, K), np.zeros(K, np.float16), padding=(0, 0)))
    dx.compile_model(m, conv_config=config, assume=assume)
    assert "nan" not in dx.last_compile_report().lower()


def test_every_configuration_has_a_measured_factor():
    """A configuration without an entry in conv_cost.cpp's table counts as slow and is hardly ever taken; one that has left the
    library would keep its entry unnoticed."""
    src = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(dx.__file__))), "denox_amd", "csrc", "compiler", "conv_cost.cpp")
    table = open(src).read().split("kFactor[] = {")[1].split("};")[0]
    names = re.findall(r'\{"(\w+)", [0-9.]+f\}', table)
    assert len(names) == len(set(names)) and set(names) == set(dx.conv_config_names()), set(names) ^ set(dx.conv_config_names())
