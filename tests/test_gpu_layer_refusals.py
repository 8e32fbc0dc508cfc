"""What the layer's one-call forms refuse, as the op-by-op forms do: caches and weights of other shapes
and types than the layer's.  Nothing is launched into a buffer that does not fit."""

from __future__ import annotations

import pytest
import torch

from ffnmem import infer
from lngram_hip import ops, workloads

pytestmark = pytest.mark.gpu


def _decode(dev, b=2, n=3):
    w = workloads.SB.with_shape(b, n)
    mem = workloads.build_memory(w, 0, dev)
    model = infer.memory_model(mem)
    h = workloads.make_hidden(w, 1, dev)
    codes = torch.randint(0, 16, (b, n, w.routes), dtype=torch.uint8, device=dev)
    return model, infer.DecodeState.empty(model, b, n + 5), h, codes


@pytest.mark.parametrize("which,shape,dtype", [("codes", (2, 8, 181), torch.uint8), ("codes", (2, 8, 200), torch.uint8),
                                               ("codes", (2, 8, 184), torch.int32), ("conv_in", (2, 8, 512), torch.bfloat16),
                                               ("conv_in", (2, 8, 2048), torch.bfloat16)])
def test_caches_of_another_layer(dev, monkeypatch, which, shape, dtype):
    model, st, h, codes = _decode(dev)
    one = []
    real = ops.memory_step
    monkeypatch.setattr(ops, "memory_step", lambda *a: one.append(1) or real(*a))
    infer.memory_step(model, 0, st, h, codes)
    assert one and real(model.blocks[0].memory.module._native_layer(h.dtype, h.device, True), h, codes, 0, st.codes[0],
                        st.conv_in[0]) is not None             # its own caches: the one call
    getattr(st, which)[0] = torch.zeros(*shape, dtype=dtype, device=dev)
    with pytest.raises((ValueError, RuntimeError)):
        infer.memory_step(model, 0, st, h, codes)
    layer = model.blocks[0].memory.module._native_layer(h.dtype, h.device, True)
    assert real(layer, h, codes, 0, st.codes[0], st.conv_in[0]) is None


def test_inputs_of_another_layer(dev):
    model, st, h, codes = _decode(dev)
    layer = model.blocks[0].memory.module._native_layer(h.dtype, h.device, True)
    for x, c in ((h[..., :512].contiguous(), codes), (h, codes[..., :100].contiguous()), (h, codes[:, :1].contiguous())):
        assert ops.memory_step(layer, x, c, 0, st.codes[0], st.conv_in[0]) is None
        with pytest.raises(ValueError, match="memory_forward"):
            ops.memory_forward(layer, x, c, 1 << 26)
    assert ops.memory_step(layer, h.float(), codes, 0, st.codes[0], st.conv_in[0]) is None
    assert ops.memory_step(layer, h, codes, 6, st.codes[0], st.conv_in[0]) is None          # past the caches
    assert ops.memory_step(layer, h, codes.cpu(), 0, st.codes[0], st.conv_in[0]) is None


@pytest.mark.parametrize("weight,shape", [("tables.ngram_2", (184 * 256 - 8, 128)), ("tables.ngram_3", (184 * 4096, 64)),
                                          ("readout_memory_norm", (128,)), ("readout_q_proj", (1024, 512)),
                                          ("readout_o_proj", (512, 1024)), ("readout_kv_proj", (512, 128)),
                                          ("short_conv.norm", (512,))])
def test_weights_of_another_layer(dev, monkeypatch, weight, shape):
    model, st, h, codes = _decode(dev)
    m = model.blocks[0].memory.module
    assert m._native_layer(h.dtype, h.device, True) is not None
    monkeypatch.setattr(ops, "memory_forward", lambda *a: pytest.fail("one call"))
    monkeypatch.setattr(ops, "memory_step", lambda *a: pytest.fail("one call"))
    m.get_submodule(weight).weight.data = torch.zeros(*shape, dtype=torch.bfloat16, device=dev)
    if weight in ("readout_q_proj", "readout_kv_proj"):        # their packed forms refuse them
        with pytest.raises(ValueError):
            m._native_layer(h.dtype, h.device, True)
    else:
        assert m._native_layer(h.dtype, h.device, True) is None
    if weight != "short_conv.norm":                            # the conv's norm weight: not checked op by op
        with pytest.raises((ValueError, RuntimeError)):
            m(h, codes)
        with pytest.raises((ValueError, RuntimeError)):
            infer.memory_step(model, 0, st, h, codes)
