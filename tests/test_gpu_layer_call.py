"""The layer's launches in one call (``lng_memory_forward``, ``lng_memory_step``) equal the op-by-op
form bit for bit, and the op-by-op form runs where the call does not stand for it."""

from __future__ import annotations

import pytest
import torch

from ffnmem import infer
from ffnmem.memory import lngram_v2
from lngram_hip import ops, workloads

pytestmark = pytest.mark.gpu

LAYERS = {
    "sb": (workloads.SB, {}), "tiny": (workloads.TINY, {}),
    "generic bf16": (workloads.MemoryWorkload("g", 96, 5, 16, 6, 3, 16, 1, 1, torch.bfloat16), {}),
}


def _layer(name, b, t, dev):
    w = LAYERS[name][0].with_shape(b, t)
    h = workloads.make_hidden(w, 1, dev)
    return workloads.build_memory(w, 0, dev), h, ops.rmsnorm(h, torch.ones(w.d_model, dtype=w.dtype, device=dev), 1e-5)


@pytest.mark.parametrize("name,b,t", [("sb", 1, 1), ("sb", 1, 65), ("sb", 3, 347), ("sb", 1, 4097), ("tiny", 4, 128),
                                      ("tiny", 1, 1), ("generic bf16", 3, 50), ("generic bf16", 2, 600)])
def test_forward_equals_the_ops(dev, monkeypatch, name, b, t):
    mem, h, hn = _layer(name, b, t, dev)
    calls = []
    real = ops.memory_forward
    monkeypatch.setattr(ops, "memory_forward", lambda *a: calls.append(1) or real(*a))
    got = mem(h, hn)
    assert calls
    mem.module._NATIVE_WORKSPACE = 0
    assert torch.equal(got, mem(h, hn))


def test_the_op_form_stays(dev, monkeypatch):
    mem, h, hn = _layer("tiny", 2, 9, dev)
    want = mem(h, hn)
    monkeypatch.setattr(ops, "memory_forward", lambda *a: pytest.fail("one call"))
    seen = []
    hook = mem.module.readout_query_norm.register_forward_hook(lambda *a: seen.append(1))
    assert torch.equal(mem(h, hn), want) and seen                       # a hook on a norm still runs
    hook.remove()
    with ops.KernelTimer("causal_conv"):
        assert torch.equal(mem(h, hn), want)                            # launches timed one by one
    mem.module.readout_o_proj.weight.data = mem.module.readout_o_proj.weight.data.double()
    with pytest.raises(AssertionError):                                 # converted per op, as before
        assert mem.module._native_layer(h.dtype, h.device, False) is not None
    assert torch.equal(mem(h, hn), want)


@pytest.mark.parametrize("b,n,length", [(1, 1, 0), (8, 1, 30), (4, 5, 11), (16, 4, 1)])
@pytest.mark.parametrize("codes_dtype", [torch.uint8, torch.int64])
def test_step_equals_the_ops(dev, monkeypatch, b, n, length, codes_dtype):
    mem, h, hn = _layer("sb", b, length + n, dev)
    model = infer.memory_model(mem)

    def run(native):
        if not native:
            monkeypatch.setattr(lngram_v2.RouteNgramMemoryV2, "_native_layer", lambda *a: None)
        st = infer.DecodeState.empty(model, b, length + n + 3)
        outs = []
        for i0, i1 in ((0, length), (length, length + n)):
            if i1 > i0:
                x = hn[:, i0:i1].contiguous()
                c = infer.memory_codes(model, 0, st, h_norm=x).to(codes_dtype)
                outs.append(infer.memory_step(model, 0, st, h[:, i0:i1].contiguous(), c))
                st.length = i1
        return outs + [st.codes[0], st.conv_in[0]]

    for x, y in zip(run(True), run(False)):
        assert torch.equal(x, y)
