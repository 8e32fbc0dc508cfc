"""``lng_memory_forward`` and ``lng_memory_step`` refuse layers that their kernels do not take, before any
GPU work (CPU)."""

from __future__ import annotations

import ctypes

import pytest
import torch

from lngram_hip import _lib
from lngram_hip.ops import dtype_code

SB = dict(hidden=1024, routes=184, bits=4, n_orders=2, mem_dim=128, q_heads=16, kv_heads=4, head_dim=64, conv_k=4,
          conv_dilation=3, fused=1)


def _layer(**change):
    L = _lib.MemoryLayer()
    for k, v in {**SB, **change}.items():
        setattr(L, k, v)
    L.orders[0], L.orders[1] = 2, 3
    L.dtype = dtype_code(torch.bfloat16)
    for f in ("w_q", "q_norm", "kv", "mem_norm", "w_o", "conv_norm", "conv_w"):
        setattr(L, f, 4096)
    L.tables[0] = L.tables[1] = 4096
    return L


def test_the_shape_that_is_served():
    lib = _lib.load()
    assert lib.lng_memory_layer_size() == ctypes.sizeof(_lib.MemoryLayer)
    assert lib.lng_memory_forward_workspace_bytes(ctypes.byref(_layer()), 2, 3) > 0


@pytest.mark.parametrize("change", [dict(hidden=512), dict(hidden=2048), dict(hidden=1024, q_heads=8), dict(mem_dim=64),
                                    dict(bits=5), dict(kv_heads=3), dict(kv_heads=0), dict(conv_k=0), dict(routes=0),
                                    dict(n_orders=5), dict(n_orders=1), dict(fused=0, hidden=96, q_heads=6, head_dim=32)])
def test_layers_that_are_refused(change):
    lib = _lib.load()
    L = _layer(**change)
    p, buf = ctypes.byref(L), ctypes.c_void_p(4096)
    assert lib.lng_memory_forward_workspace_bytes(p, 2, 3) == 0
    assert lib.lng_memory_forward(p, buf, buf, dtype_code(torch.uint8), 2, 3, buf, 1 << 40, buf, None) == -1
    assert b"memory_forward" in lib.lng_last_error()
    assert lib.lng_memory_step(p, buf, buf, dtype_code(torch.uint8), 2, 3, 0, buf, buf, 8, buf, 1 << 40, buf, None) == -1
    assert b"memory_step" in lib.lng_last_error()


@pytest.mark.parametrize("args", [dict(n=40), dict(n=-1), dict(pos0=-1), dict(pos0=6), dict(nws=100), dict(codes=None)])
def test_steps_that_are_refused(args):
    lib = _lib.load()
    a = {"n": 3, "pos0": 0, "nws": 1 << 40, "codes": 4096, **args}
    buf = ctypes.c_void_p(4096)
    rc = lib.lng_memory_step(ctypes.byref(_layer()), buf, a["codes"], dtype_code(torch.uint8), 2, a["n"], a["pos0"], buf, buf, 8, buf,
                             a["nws"], buf, None)
    assert rc == -1 and b"memory_step" in lib.lng_last_error()
