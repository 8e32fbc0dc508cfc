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
    assert one == [1]                                          # its own caches: the one call
    getattr(st, which)[0] = torch.zeros(*shape, dtype=dtype, device=dev)
    with pytest.raises((ValueError, RuntimeError)):
        infer.memory_step(model, 0, st, h, codes)
    assert one == [1]
    layer = model.blocks[0].memory.module._native_layer(h.dtype, h.device, True)
    with pytest.raises(ValueError, match="code cache"):
        real(layer, h, codes, 0, st.codes[0], st.conv_in[0])


def test_inputs_of_another_layer(dev):
    model, st, h, codes = _decode(dev)
    layer = model.blocks[0].memory.module._native_layer(h.dtype, h.device, True)
    for x, c in ((h[..., :512].contiguous(), codes), (h, codes[..., :100].contiguous()), (h, codes[:, :1].contiguous())):
        with pytest.raises(ValueError, match="code cache"):
            ops.memory_step(layer, x, c, 0, st.codes[0], st.conv_in[0])
