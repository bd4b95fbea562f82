"""Instances of at most four dispatches launch them one by one, longer ones replay a captured graph: the same bits from both, with more
sets of interface addresses than graphs are kept, as a frame sequence, and with the graph switched off."""
import numpy as np
import pytest

import denox_amd as dx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dispatches", [1, 4, 5, 8])
def test_few_dispatches(dispatches, monkeypatch):
    torch = pytest.importorskip("torch")
    H, W, C = 36, 52, 8
    m = dx.Model()
    t = m.input("input", "W", "H", C)
    for _ in range(dispatches // 2):
        t = m.pool(m.upsample(t))  # the identity, whole numbers of bits
    if dispatches % 2:
        t = m.pool(t)
    m.output(t)
    mod = dx.Module.compile(m)
    assert mod.runtime_model.dispatch_count == dispatches
    rng = np.random.default_rng(dispatches)
    xs = [rng.standard_normal((H, W, C)).astype(np.float16) for _ in range(6)]
    wants = [x.reshape(H // 2, 2, W // 2, 2, C).max((1, 3)) if dispatches % 2 else x for x in xs]
    inst = mod.instance(H=H, W=W)
    monkeypatch.setenv("DENOX_HIP_NO_GRAPH", "1")
    plain = mod.instance(H=H, W=W)
    d_in = [torch.from_numpy(x).cuda() for x in xs]
    for i in (inst, plain):
        outs = [torch.zeros(w.shape, dtype=torch.float16, device="cuda") for w in wants]
        torch.cuda.synchronize()
        for x, o in zip(d_in, outs):
            i.infer_device([x.data_ptr()], [o.data_ptr()])
        i.synchronize()
        for o, w in zip(outs, wants):
            np.testing.assert_array_equal(o.cpu().numpy(), w)
        for got, w in zip(i.infer_many([[x] for x in xs]), wants):
            np.testing.assert_array_equal(got[0], w)
        np.testing.assert_array_equal(i.infer(xs[0])[0], wants[0])
