"""Schedules selected without a timing table: what the estimates may decide and what they leave to a caller's table or to a name."""
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
