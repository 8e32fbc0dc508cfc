"""A token's fused readout has the same bits whatever launch it is part of: alone or among few tokens (its
routes over eight waves), in a launch's remainder (over four), in a whole round of blocks (one wave), from
the codes of its sequence, of a cache or of its own window, and as given rows."""

from __future__ import annotations

import math

import pytest
import torch

from lngram_hip import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [1, 31, 33, 64, 129, 184, 225, 256])
@pytest.mark.parametrize("std", [3.0, 100.0])      # 100: the running maximum moves in most chunks
def test_every_form_gives_the_same_bits(dev, R, std):
    gen = torch.Generator(device=dev).manual_seed(R)

    def rnd(*shape, std):
        return (torch.randn(*shape, generator=gen, device=dev) * std).to(torch.bfloat16)

    T = 2561                                        # one whole round of 2048 tokens and past 512 more
    t2, t3, kv, wm = rnd(R * 256, 128, std=0.02), rnd(R * 4096, 128, std=0.02), rnd(512, 256, std=0.05), rnd(256, std=1.0)
    q, h = rnd(1, T, 1024, std=std), rnd(1, T, 1024, std=1.0)
    codes = torch.randint(0, 16, (1, T, R), generator=gen, device=dev, dtype=torch.uint8)
    args = (ops.memory_readout_pack(kv), wm, 1e-5, 0.125, math.log(R) if R > 1 else 0.5)
    qk = {"q_rows": h, "q_eps": 1e-5}
    whole = ops.memory_readout_fused(q, codes, t2, t3, *args, **qk)     # 2561: every token in an unsplit block
    assert torch.isfinite(whole.float()).all()
    for n in (1, 5, 256, 257, 512, 513, 2048, 2049, 2304, 2560):        # both sides of the forms' lines
        got = ops.memory_readout_fused_at(q[:, T - n:].contiguous(), codes, T - n, t2, t3, *args,
                                          q_rows=h[:, T - n:].contiguous(), q_eps=1e-5)
        assert torch.equal(got, whole[:, T - n:]), n
    for n in (16, 300):
        win = torch.stack([codes[0, T - n - 2 + k:T - 2 + k] for k in range(3)], 1).contiguous()
        seg, val = torch.zeros(n, 3, dtype=torch.int32, device=dev), torch.ones(n, 3, dtype=torch.uint8, device=dev)
        tail = (q[:, T - n:].contiguous(),)
        kw = {"q_rows": h[:, T - n:].contiguous(), "q_eps": 1e-5}
        assert torch.equal(ops.memory_readout_fused_windows(*tail, win, seg, val, t2, t3, *args, **kw), whole[:, T - n:])
        rows = ops.route_tokens(codes, [t2, t3], (2, 3), 4, target_length=n)
        assert torch.equal(ops.memory_readout_fused_rows(*tail, rows, *args, **kw), whole[:, T - n:])


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_values_that_are_not_finite_stay_in_their_token(dev, bad):
    R, T = 184, 300
    gen = torch.Generator(device=dev).manual_seed(1)

    def rnd(*shape, std):
        return (torch.randn(*shape, generator=gen, device=dev) * std).to(torch.bfloat16)

    args = (rnd(R * 256, 128, std=0.02), rnd(R * 4096, 128, std=0.02), ops.memory_readout_pack(rnd(512, 256, std=0.05)),
            rnd(256, std=1.0), 1e-5, 0.125, math.log(R))
    q = rnd(1, T, 1024, std=3.0)
    codes = torch.randint(0, 16, (1, T, R), generator=gen, device=dev, dtype=torch.uint8)
    for n in (200, 300):                            # eight waves a token; four
        c, x = codes[:, :n].contiguous(), q[:, :n].clone()
        want = ops.memory_readout_fused(x, c, *args)
        x[0, 100, 7] = bad
        got = ops.memory_readout_fused(x, c, *args)
        assert not torch.isfinite(got[0, 100].float()).all()
        got[0, 100] = want[0, 100]
        assert torch.equal(got, want)


def test_trees_of_many_sequences_equal_their_chains(dev):
    """Draft-tree verification of 17 sequences (272 nodes: past the one-token blocks of the readout and the
    skinny projections) against chain decodes of 17 rows, bit for bit."""
    from drafting.tree import tree16
    from ffnmem.infer import DecodeState, memory_codes, memory_model, memory_step, tree_memory_step
    from lngram_hip import workloads as wl

    parent, b, L = tree16().parent, 17, 5
    n = len(parent)
    w = wl.SB.with_shape(b, L + n)
    mem, h = wl.build_memory(w, seed=0, device=dev), wl.make_hidden(w, seed=1, device=dev)
    h_norm = ops.rmsnorm(h, torch.ones(w.d_model, dtype=w.dtype, device=dev), w.norm_eps)
    model, rows = memory_model(mem), torch.arange(b, device=dev)
    with torch.no_grad():
        st = DecodeState.empty(model, b, L + n)
        memory_step(model, 0, st, h[:, :L].contiguous(), memory_codes(model, 0, st, h_norm=h_norm[:, :L].contiguous()))
        st.length = L
        base = st.index_select(rows)
        hn = h[:, L:].contiguous()
        codes = memory_codes(model, 0, st, h_norm=h_norm[:, L:].contiguous())
        got = tree_memory_step(model, 0, st, hn, codes, parent)
        for i in (0, 3, n - 1):
            path = [i]
            while parent[path[0]] >= 0:
                path.insert(0, parent[path[0]])
            sti = base.index_select(rows)
            for p in path:
                out = memory_step(model, 0, sti, hn[:, p:p + 1].contiguous(), codes[:, p:p + 1].contiguous())
                sti.length += 1
            assert torch.equal(got[:, i:i + 1], out), i
