"""The work that users of this library give it, as measurable cases.

A case is one pass through public entry points at stated sizes: the memory layer over whole
sequences (bf16 SB / SD-C layers, the fp32 tiny layer), its cached decode and verification steps,
the drafter's tree and chain steps, the training lookup with its backward, and the scaled-table
gather.  ``listed()`` holds the named ones, ``draw(rng)`` gives others of the same ranges,
``prepare`` builds what a program holds before the call, ``run`` is one pass, ``work`` the bytes
and operations that it cannot do without, ``exact`` the same result in 64 bits by plain torch.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parent.parent / "lngram-decode_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

D, MEM, QH, KVH, HD, BITS, EPS = 1024, 128, 16, 4, 64, 4, 1e-5   # the SB / SD layers
ORDERS = (2, 3)
VOCAB, SSM = 32768, 256


# ----------------------------------------------------------------------------- the cases
def listed() -> list:
    return [
        # the SB layer over a training-size or batched-prefill batch: the headline configuration
        {"name": "prefill_8x2048", "kind": "prefill", "batch": 8, "seq": 2048, "routes": 184},
        # a few prompts of an odd length prefilled together
        {"name": "prefill_3x777", "kind": "prefill", "batch": 3, "seq": 777, "routes": 184},
        # one short prompt: the time to the first token
        {"name": "prefill_1x200", "kind": "prefill", "batch": 1, "seq": 200, "routes": 184},
        # the SD-C layer with its SSM and token router, whole batch of long sequences
        {"name": "sdc_8x4096", "kind": "sdc", "batch": 8, "seq": 4096, "routes": 181},
        # the CPU-scale fp32 layer of experiments and tests: launches and latency count
        {"name": "tiny_fp32_4x128", "kind": "tiny", "batch": 4, "seq": 128},
        # serving: one new token of each of 8 sequences, replayed from a captured graph
        {"name": "decode_8x1", "kind": "decode", "batch": 8, "new": 1, "cached": 2048},
        # verification of a drafted chain (4 drafts + 1) for 4 sequences, launched eagerly
        {"name": "verify_4x5", "kind": "verify", "batch": 4, "new": 5, "cached": 1000},
        # verification of the 16-node draft tree of one sequence, replayed from a captured graph
        {"name": "tree_verify_16", "kind": "tree_verify", "nodes": 16, "cached": 2048},
        # the SD-B drafter's tree step with online counts and its verification gather
        {"name": "draft_tree_16", "kind": "draft_tree", "nodes": 16, "context": 2048, "online": True},
        # the SD-C drafter's live step: commit the accepted tokens, draft 4 over the sketch shortlist
        {"name": "draft_chain_sdc", "kind": "draft_chain", "model": "sdc", "sketch": True, "context": 256,
         "commit": 2, "gamma": 4},
        # training: the lookup with its surrogate, forward and backward (logits' and tables' gradients)
        {"name": "train_lookup_8x2048", "kind": "train", "batch": 8, "seq": 2048, "routes": 184},
        # the tables grown 64 times (13 GB): random rows from memory past every cache
        {"name": "scaled_16x4096", "kind": "scaled", "batch": 16, "seq": 4096, "routes": 184, "scale_log2": 6},
    ]


def _log(rng, lo: int, hi: int) -> int:
    """An integer of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _batch_seq(rng, most: int, max_batch: int) -> tuple:
    """Sequences of at least 3 positions, the first that every order's rows reach."""
    b = _log(rng, 1, max_batch)
    return b, _log(rng, 3, most // b)


def draw(rng) -> dict:
    kind = rng.choice(("prefill", "prefill", "sdc", "tiny", "decode", "verify", "tree_verify", "draft_tree",
                       "draft_chain", "train", "train", "scaled"))
    if kind == "prefill":
        b, t = _batch_seq(rng, 16384, 16)
        return {"kind": kind, "batch": b, "seq": t, "routes": rng.choice((181, 182, 184))}
    if kind == "sdc":
        b, t = _batch_seq(rng, 32768, 8)
        return {"kind": kind, "batch": b, "seq": t, "routes": 181}
    if kind == "tiny":
        b, t = _batch_seq(rng, 4096, 8)
        return {"kind": kind, "batch": b, "seq": t}
    if kind in ("decode", "verify"):
        new = rng.randint(1, 6)
        return {"kind": kind, "batch": _log(rng, 1, 64 // new), "new": new, "cached": _log(rng, 1, 4096)}
    if kind == "tree_verify":
        return {"kind": kind, "nodes": rng.choice((8, 16)), "cached": _log(rng, 1, 4096)}
    if kind == "draft_tree":
        return {"kind": kind, "nodes": rng.choice((8, 16)), "context": _log(rng, 8, 3000),
                "online": rng.random() < 0.5}
    if kind == "draft_chain":
        model = rng.choice(("sdb", "sdc"))
        return {"kind": kind, "model": model, "sketch": model == "sdc" and rng.random() < 0.5,
                "context": _log(rng, 8, 2048), "commit": rng.randint(1, 5), "gamma": rng.randint(1, 6)}
    if kind == "train":
        b, t = _batch_seq(rng, 16384, 16)
        return {"kind": kind, "batch": b, "seq": t, "routes": rng.choice((181, 182, 184))}
    b, t = _batch_seq(rng, 65536, 16)
    return {"kind": kind, "batch": b, "seq": t, "routes": rng.choice((181, 184)), "scale_log2": rng.randint(2, 6)}


# ----------------------------------------------------------------------------- inputs
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _randn(g, *shape, std=1.0, dtype=torch.float32) -> torch.Tensor:
    return torch.empty(*shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=g)


def _randint(g, hi: int, *shape, dtype=torch.int64) -> torch.Tensor:
    return torch.randint(0, hi, shape, generator=g, device="cuda", dtype=dtype)


def _memory(seed: int, cfg: dict, d: int, dtype, ssm: int = 0):
    """An ``LngramMemory`` in eval mode with drawn weights (the zero-initialised output projection
    and conv too, so that the output depends on the memory)."""
    from ffnmem.memory.wrapper import LngramMemory

    torch.manual_seed(int(seed) + 101)
    with torch.device("cuda"):
        mem = LngramMemory(d, dict(cfg, execution_mode="full"), init_std=0.02, norm_eps=EPS, ssm_dim=ssm)
        m = mem.module
        with torch.no_grad():
            m.readout_o_proj.weight.normal_(0.0, 0.02)
            m.short_conv.conv.weight.normal_(0.0, 0.2)
    return mem.to(dtype).eval()


def _sb_cfg(routes: int) -> dict:
    return {"routes": routes, "mem_dim": MEM, "kv_heads": KVH, "q_heads": QH, "head_dim": HD}


def _unit_norm(h: torch.Tensor) -> torch.Tensor:
    """The block's normalised hidden states, as its pre-norm hands them to the router."""
    f = h.float()
    return (f * torch.rsqrt(f.pow(2).mean(-1, keepdim=True) + EPS)).to(h.dtype)


def _tree_spec(nodes: int):
    from drafting.tree import default_tree, tree16

    return tree16() if nodes == 16 else default_tree()


def _bundle(case: dict, seed: int) -> tuple:
    """(config, tensors) of a drafter: weights ~N(0, 0.02), bf16, norms one."""
    from lngram_hip.workloads import SDB_DRAFT, SDC_DRAFT

    g = _gen(seed)
    w = SDC_DRAFT if case.get("model") == "sdc" else SDB_DRAFT
    cfg, n, r = w.config(), w.ssm_dim, w.routes
    bf = torch.bfloat16

    def rnd(*shape):
        return _randn(g, *shape, std=0.02, dtype=bf)

    def ones(k):
        return torch.ones(k, dtype=bf, device="cuda")

    inner, kh = w.q_heads * w.head_dim, w.kv_heads * w.head_dim
    t = {"embedding": rnd(w.vocab, D), "table_2": rnd(r * 16 ** 2, MEM), "table_3": rnd(r * 16 ** 3, MEM),
         "mem_norm": ones(2 * MEM), "kv_proj": rnd(2 * kh, 2 * MEM), "router": rnd(4 * r, 2 * D + n),
         "router_prev_norm": ones(D), "router_cur_norm": ones(D), "router_start": rnd(D), "q_norm": ones(D),
         "w_q": rnd(inner, D), "w_o": rnd(D, inner), "out_norm": ones(D)}
    if n:
        t["ssm_norm"], t["ssm_w_in"], t["w_sq"] = ones(D), rnd(n, D), rnd(inner, n)
        t["ssm_decay"] = 0.9 + 0.099 * torch.rand(n, generator=g, device="cuda")
    if case.get("sketch"):
        for o in ORDERS:
            t[f"sketch_ids_{o}"] = _randint(g, VOCAB, r * 16 ** o, 16, dtype=torch.int32)
            t[f"sketch_counts_{o}"] = _randint(g, 4, r * 16 ** o, 16)
        t["fallback"] = torch.randperm(VOCAB, generator=g, device="cuda")[:64].to(torch.int32)
        cfg = dict(cfg, sketch_k=16, shortlist_cap=64)
    toks = _randint(g, VOCAB, case["context"] + case.get("commit", 0)).tolist()
    return cfg, t, toks


def _cached(case: dict, seed: int, batch: int, new: int) -> dict:
    """An SB layer with ``cached`` positions decoded, and the hidden states of ``new`` more."""
    from ffnmem.infer import DecodeState, memory_codes, memory_model, memory_step

    L = case["cached"]
    mem = _memory(seed, _sb_cfg(184), D, torch.bfloat16)
    model = memory_model(mem)
    h = _randn(_gen(seed), batch, L + new, D).to(torch.bfloat16)
    hn = _unit_norm(h)
    st = DecodeState.empty(model, batch, L + 16)
    with torch.no_grad():
        memory_step(model, 0, st, h[:, :L].contiguous(), memory_codes(model, 0, st, h_norm=hn[:, :L].contiguous()))
    st.length = L
    return {"mem": mem, "model": model, "st": st, "all_h": h, "all_hn": hn, "h": h[:, L:].contiguous(),
            "hn": hn[:, L:].contiguous(), "L_t": torch.full((), L, dtype=torch.int32, device="cuda")}


def _capture(step) -> tuple:
    """(graph, output) of a step captured once, as a serving loop keeps it."""
    with torch.no_grad():
        step()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = step()
    return graph, out


def prepare(case: dict, seed: int) -> dict:
    kind, s = case["kind"], {"case": case}
    g = _gen(seed)
    if kind == "prefill":
        s["mem"] = _memory(seed, _sb_cfg(case["routes"]), D, torch.bfloat16)
        s["h"] = _randn(g, case["batch"], case["seq"], D).to(torch.bfloat16)
        s["hn"] = _unit_norm(s["h"])
    elif kind == "tiny":
        s["mem"] = _memory(seed, {"routes": 8, "mem_dim": 32, "kv_heads": 2, "q_heads": 4, "head_dim": 32}, 128,
                           torch.float32)
        s["h"] = _randn(g, case["batch"], case["seq"], 128)
        s["hn"] = _unit_norm(s["h"])
    elif kind == "sdc":
        from ffnmem.memory.ssm import DiagonalSSM

        b, t = case["batch"], case["seq"]
        s["mem"] = _memory(seed, dict(_sb_cfg(case["routes"]), router_input="embed2_ssm"), D, torch.bfloat16, SSM)
        with torch.device("cuda"):
            s["ssm"] = DiagonalSSM(D, SSM).eval()        # fp32, beside the bf16 layers
        s["emb_table"] = _randn(g, VOCAB, D, std=0.02).to(torch.bfloat16)
        s["tok"] = _randint(g, VOCAB, b, t)
        s["emb"] = s["emb_table"][s["tok"]]              # the model's input embeddings, which it has anyway
        s["h"] = _randn(g, b, t, D).to(torch.bfloat16)
        s["mem"].router_features.tables(s["emb_table"])  # once per weight version
    elif kind == "decode":
        from ffnmem.infer import static_memory_step

        s.update(_cached(case, seed, case["batch"], case["new"]))
        s["graph"], s["out"] = _capture(
            lambda: static_memory_step(s["model"], 0, s["st"], s["h"], None, s["L_t"], router_x=s["hn"]))
    elif kind == "verify":
        s.update(_cached(case, seed, case["batch"], case["new"]))
    elif kind == "tree_verify":
        from ffnmem.infer import memory_codes, static_tree_memory_step

        s.update(_cached(case, seed, 1, case["nodes"]))
        parent = _tree_spec(case["nodes"]).parent
        s["graph"], s["out"] = _capture(lambda: static_tree_memory_step(
            s["model"], 0, s["st"], s["h"], memory_codes(s["model"], 0, s["st"], h_norm=s["hn"]), parent, s["L_t"]))
    elif kind in ("draft_tree", "draft_chain"):
        from drafting.gpu_drafter import GpuDrafter

        cfg, t, toks = _bundle(case, seed)
        dr = GpuDrafter((cfg, t), device=torch.device("cuda", torch.cuda.current_device()), max_len=len(toks) + 16,
                        online=bool(case.get("online")))
        n = case["context"]
        dr.commit(toks[:n])
        s.update(drafter=dr, next=toks[n:], spec=_tree_spec(case["nodes"]) if kind == "draft_tree" else None)
        if kind == "draft_tree":
            dr.tree_step(s["spec"], graph=True)          # captured once per tree shape
    elif kind == "train":
        b, t, r = case["batch"], case["seq"], case["routes"]
        s["mem"] = _memory(seed, _sb_cfg(r), D, torch.bfloat16).train()
        s["codes"] = _randint(g, 16, b, t, r, dtype=torch.uint8)
        # route logits whose signs are the codes, as the router that made them gives
        bit = (s["codes"][..., None] >> torch.arange(BITS, device="cuda", dtype=torch.uint8)) & 1
        s["q"] = (_randn(g, b, t, r, BITS).abs() * (bit.float() * 2 - 1)).requires_grad_(True)
        s["grad"] = _randn(g, b, t, r, 2 * MEM, std=0.01, dtype=torch.bfloat16)
    elif kind == "scaled":
        b, t, r, sl = case["batch"], case["seq"], case["routes"], case["scale_log2"]
        s["tables"] = [_randn(g, r << (sl + BITS * o), MEM, std=0.02, dtype=torch.bfloat16) for o in ORDERS]
        s["codes"] = _randint(g, 16, b, t, r, dtype=torch.uint8)
        s["seed"] = (seed * 2654435761 + 12345) & 0xFFFFFFFF
    else:
        raise ValueError(kind)
    return s


# ----------------------------------------------------------------------------- one pass
def run(s: dict):
    kind = s["case"]["kind"]
    if kind == "train":
        m = s["mem"].module
        tables = [m.tables[f"ngram_{o}"].weight for o in ORDERS]
        rows = m._lookup_route_chunk(s["codes"], s["q"], 0, m.num_routes, None, None)
        gq, g2, g3 = torch.autograd.grad(rows, [s["q"], *tables], s["grad"])
        return {"rows": rows.detach(), "grad_q": gq, "grad_2": g2, "grad_3": g3}
    with torch.no_grad():
        if kind in ("prefill", "tiny"):
            return s["mem"](s["h"], s["hn"])
        if kind == "sdc":
            states = s["ssm"](s["emb"])
            return {"states": states, "out": s["mem"].forward_ids(s["h"], s["tok"], s["emb_table"], states)}
        if kind in ("decode", "tree_verify"):
            s["graph"].replay()
            return {"out": s["out"], "codes": s["st"].codes[0], "conv_in": s["st"].conv_in[0]}
        if kind == "verify":
            from ffnmem.infer import memory_decode

            out = memory_decode(s["model"], 0, s["st"], s["h"], h_norm=s["hn"])
            return {"out": out, "codes": s["st"].codes[0], "conv_in": s["st"].conv_in[0]}
        if kind == "draft_tree":
            tokens, rows = s["drafter"].tree_step(s["spec"], graph=True)
            return {"tokens": tokens, "rows": rows}
        if kind == "draft_chain":
            dr = s["drafter"]
            n = dr.length
            dr.commit(s["next"])
            out = dr.draft(s["case"]["gamma"])
            dr.truncate(n)
            return {"ids": out.topk_ids, "logits": out.topk_logits, "codes": out.codes}
        if kind == "scaled":
            from lngram_hip import ops

            return ops.gather_sum_scaled(s["tables"], s["codes"], ORDERS, BITS, s["case"]["scale_log2"], s["seed"])
    raise ValueError(kind)


# ----------------------------------------------------------------------------- the least work
def _distinct(rows: float, reads: float) -> float:
    """Expected distinct rows met by so many uniform reads."""
    return rows * -math.expm1(reads * math.log1p(-1.0 / rows))


def _row_bytes(n: int, routes: int, scale: int = 1, width: int = 2 * MEM) -> float:
    return sum(routes * width * _distinct(scale * 16.0 ** o, n) for o in ORDERS)


def _readout_flops(n: int, routes: int) -> float:
    # q -> key space, scores and weighted rows over the routes, value projection of 16 heads
    return 2.0 * n * QH * (HD * 2 * MEM + 2 * routes * 2 * MEM + 2 * MEM * HD)


def _layer_work(n: int, routes: int, feat: int) -> dict:
    weights = 2.0 * (4 * routes * feat + 2 * D * D + 2 * KVH * HD * 2 * MEM)
    return {"bytes": n * 2.0 * (D + D) + _row_bytes(n, routes) + weights,
            "flops": 2.0 * n * (4 * routes * feat + 2 * D * D) + _readout_flops(n, routes)}


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("prefill", "decode", "verify", "tree_verify"):
        n = case["nodes"] if kind == "tree_verify" else case["batch"] * case["seq" if kind == "prefill" else "new"]
        w = _layer_work(n, case.get("routes", 184), D)
        w["bytes"] += 2.0 * n * D                        # h_norm beside h
        return w
    if kind == "sdc":
        n = case["batch"] * case["seq"]
        w = _layer_work(n, case["routes"], 2 * D + SSM)
        emb = 2.0 * D * _distinct(VOCAB, n)
        return {"bytes": w["bytes"] + emb + n * 4.0 * SSM + 2.0 * n * D + 4.0 * SSM * D,
                "flops": w["flops"] + 2.0 * n * SSM * D}
    if kind == "tiny":
        n = case["batch"] * case["seq"]
        return {"bytes": 4.0 * (3 * n * 128 + 8 * 32 * sum(_distinct(16.0 ** o, n) for o in ORDERS)
                                + 128 * (32 + 256) + 64 * 128),
                "flops": 2.0 * n * (128 * (32 + 256) + 4 * (32 * 64 + 2 * 8 * 64 + 64 * 32))}
    if kind == "draft_tree":
        # the scored positions' logits need the vocabulary table once per step (folded with the output
        # projection: 256 columns), and every node's rows are read and handed out
        inner, r = 256, 182
        return {"bytes": 4.0 * VOCAB * inner + 2.0 * case["nodes"] * r * 2 * 2 * MEM,
                "flops": 2.0 * 10 * VOCAB * inner}
    if kind == "draft_chain":
        n, r = case["commit"] + case["gamma"], 182
        feat = 2 * D + (SSM if case["model"] == "sdc" else 0)
        vocab = 64 * D * 2.0 * case["gamma"] if case["sketch"] else 2.0 * VOCAB * D
        return {"bytes": 2.0 * 4 * r * feat + 2.0 * 2 * 256 * D + vocab + n * r * 2 * 2.0 * MEM,
                "flops": 2.0 * n * (4 * r * feat + 2 * 256 * D)
                + 2.0 * case["gamma"] * D * (64 if case["sketch"] else VOCAB)}
    if kind == "train":
        n, r = case["batch"] * case["seq"], case["routes"]
        tables = sum(2.0 * MEM * r * 16 ** o for o in ORDERS)
        return {"bytes": _row_bytes(n, r) + 2 * (n * r * 2.0 * 2 * MEM) + n * r * (1 + 2 * 4.0 * BITS) + tables,
                "flops": 2.0 * n * r * MEM * sum(BITS * o + 2 for o in ORDERS)}
    n, r = case["batch"] * case["seq"], case["routes"]
    return {"bytes": _row_bytes(n, r, 1 << case["scale_log2"]) + n * (r + 4.0 * MEM), "flops": 1.0 * n * r * 2 * MEM}


def tolerance(case: dict):
    kind = case["kind"]
    if kind in ("prefill", "sdc", "decode", "verify", "tree_verify"):
        # bf16 roundings along the layer; a route logit within rounding of zero may change its sign,
        # and with it one of a token's 184 rows
        return {"rel": 1e-2, "max": 0.5, "differ": 1e-3}
    if kind == "tiny":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "draft_tree":
        return "exact"
    if kind == "draft_chain":
        return {"rel": 2e-5, "max": 1e-3, "differ": 0.0}
    if kind == "train":
        return {"rel": 4e-3, "max": 4e-2}                # bf16 table gradients: a rounding of fp32 sums
    return {"rel": 1e-6, "max": 1e-4}                    # fp32 sums of 368 rows


# ----------------------------------------------------------------------------- the same in 64 bits
def _rms64(x: torch.Tensor, w, eps: float) -> torch.Tensor:
    y = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w.double()


def _pack64(logits: torch.Tensor) -> torch.Tensor:
    b = (logits > 0).view(*logits.shape[:-1], -1, BITS).long()
    return (b << torch.arange(BITS, device=b.device)).sum(-1)


def _rows64(tables, codes: torch.Tensor) -> torch.Tensor:
    """[B, T, R, len * mem] float64 rows of codes [B, T, R] (zero before position order - 1)."""
    b, t, r = codes.shape
    base = torch.arange(r, device=codes.device)
    parts = []
    for o, tab in zip(ORDERS, tables):
        out = torch.zeros(b, t, r, tab.shape[1], dtype=torch.float64, device=codes.device)
        if t >= o:
            addr = sum(codes[:, k:t - o + 1 + k] << (BITS * k) for k in range(o))
            out[:, o - 1:] = tab[base * 16 ** o + addr].double()
        parts.append(out)
    return torch.cat(parts, -1)


def _mixed64(m, h: torch.Tensor, codes: torch.Tensor) -> torch.Tensor:
    """Output projection of the sink readout, float64 [B, T, d], one sequence and 128 positions at a time."""
    b, t, d = h.shape
    tabs = [m.tables[f"ngram_{o}"].weight.detach() for o in ORDERS]
    kvw, wo, wq = (x.weight.detach().double() for x in (m.readout_kv_proj, m.readout_o_proj, m.readout_q_proj))
    nkv, hd, grp = m.readout_num_kv_heads, m.readout_head_dim, m.readout_groups
    r = codes.shape[-1]
    out = torch.empty(b, t, d, dtype=torch.float64, device=h.device)
    for i in range(b):
        for t0 in range(0, t, 128):
            t1, a = min(t, t0 + 128), max(0, t0 - 2)
            tok = _rows64(tabs, codes[i:i + 1, a:t1])[0, t0 - a:]
            n = t1 - t0
            kv = _rms64(tok, m.readout_memory_norm.weight, m.readout_memory_norm.eps).reshape(n * r, -1) @ kvw.t()
            kv = kv.view(n, r, 2, nkv, hd)
            key = kv[:, :, 0].permute(0, 2, 1, 3).contiguous()
            val = kv[:, :, 1].permute(0, 2, 1, 3).contiguous()
            q = _rms64(h[i, t0:t1].double(), m.readout_query_norm.weight, m.readout_query_norm.eps) @ wq.t()
            sc = (q.view(n, nkv, grp, 1, hd) * key[:, :, None]).sum(-1) * hd ** -0.5
            full = torch.cat((sc, torch.full_like(sc[..., :1], math.log(r))), -1)
            p = torch.softmax(full, -1)[..., :-1]
            head = (p[..., None] * val[:, :, None]).sum(-2).reshape(n, -1)
            out[i, t0:t1] = head @ wo.t()
    return out


def _conv64(m, mixed: torch.Tensor) -> torch.Tensor:
    conv = m.short_conv
    x = _rms64(mixed, conv.norm.weight, conv.norm.eps)
    w = conv.conv.weight.detach().double()[:, 0]
    y = torch.zeros_like(x)
    t, k = x.shape[1], w.shape[1]
    for j in range(k):
        back = (k - 1 - j) * conv.dilation
        if back < t:
            y[:, back:] += x[:, :t - back] * w[:, j]
    return mixed + y * torch.sigmoid(y)


def _layer64(mem, h: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    codes = torch.cat([_pack64(x[i:i + 1].double() @ mem.router.weight.detach().double().t())
                       for i in range(x.shape[0])])
    return _conv64(mem.module, _mixed64(mem.module, h, codes))


def _scan64(ssm, emb: torch.Tensor) -> torch.Tensor:
    a = torch.sigmoid(ssm.theta.detach().float()).double()
    u = torch.stack([_rms64(e.double(), ssm.norm.weight.detach(), ssm.norm.eps)
                     @ ssm.w_in.weight.detach().double().t() for e in emb])
    u = u * (1 - a)
    out, state = torch.empty_like(u), torch.zeros_like(u[:, 0])
    for i in range(u.shape[1]):
        state = a * state + u[:, i]
        out[:, i] = state
    return out


def _chain64(case: dict, seed: int) -> dict:
    """Top-k logits of the greedy chain: the drafter's per-token algorithm in float64."""
    cfg, t, toks = _bundle(case, seed)
    dev = torch.device("cuda")
    r, n, n_kv, hd, k = cfg["routes"], cfg["ssm_dim"], cfg["kv_heads"], cfg["head_dim"], 3
    w = {x: v.double() for x, v in t.items() if v.is_floating_point() and x not in ("embedding", "table_2", "table_3")}
    emb, rows0 = t["embedding"], torch.arange(r, device=dev)
    grp = cfg["q_heads"] // n_kv
    state = torch.zeros(max(n, 1), dtype=torch.float64, device=dev)
    ids = torch.tensor(toks, device=dev)
    if n:
        u = _rms64(emb[ids].double(), w["ssm_norm"], cfg["ssm_eps"]) @ w["ssm_w_in"].t()
    states = []
    for i in range(len(toks) if n else 0):
        state = w["ssm_decay"] * state + (1 - w["ssm_decay"]) * u[i]
        states.append(state)

    def code(prev, cur, st):
        p = emb[prev].double() if prev is not None else w["router_start"]
        f = [_rms64(p, w["router_prev_norm"], cfg["router_eps"]),
             _rms64(emb[cur].double(), w["router_cur_norm"], cfg["router_eps"])] + ([st] if n else [])
        return _pack64((w["router"] @ torch.cat(f))[None])[0]

    hist = [code(toks[i - 1] if i else None, toks[i], states[i] if n else None)
            for i in range(max(0, len(toks) - 3), len(toks))]
    pos, cur, out = len(toks), toks[-1], []
    for step in range(case["gamma"]):
        rows, tok = {}, []
        for o in ORDERS:
            if pos < o:
                tok.append(torch.zeros(r, MEM, dtype=torch.float64, device=dev))
                continue
            rows[o] = rows0 * 16 ** o + sum(hist[len(hist) - o + j] << (BITS * j) for j in range(o))
            tok.append(t[f"table_{o}"][rows[o]].double())
        kv = (_rms64(torch.cat(tok, -1), w["mem_norm"], cfg["mem_eps"]) @ w["kv_proj"].t()).view(r, 2, n_kv, hd)
        q = w["w_q"] @ _rms64(emb[cur].double(), w["q_norm"], cfg["draft_eps"])
        if n:
            q = q + w["w_sq"] @ states[-1]
        sc = (q.view(n_kv, grp, 1, hd) * kv[:, 0].permute(1, 0, 2)[:, None]).sum(-1) * cfg["softmax_scale"]
        p = torch.softmax(torch.cat((sc, torch.full_like(sc[..., :1], cfg["sink_logit"])), -1), -1)[..., :-1]
        head = (p[..., None] * kv[:, 1].permute(1, 0, 2)[:, None]).sum(-2).reshape(-1)
        hid = _rms64(w["w_o"] @ head, w["out_norm"], cfg["draft_eps"])
        cand = torch.arange(VOCAB, device=dev)
        if case["sketch"]:
            tot = torch.zeros(VOCAB, dtype=torch.int64, device=dev)
            for o in rows:
                tot.index_add_(0, t[f"sketch_ids_{o}"][rows[o]].reshape(-1).long(),
                               t[f"sketch_counts_{o}"][rows[o]].reshape(-1))
            tot = tot.cpu().numpy()
            named = np.flatnonzero(tot > 0)
            sl = [int(x) for x in named[np.lexsort((named, -tot[named]))][:cfg["shortlist_cap"]]]
            for f in t["fallback"].tolist():
                if len(sl) < cfg["shortlist_cap"] and f not in sl:
                    sl.append(f)
            cand = torch.tensor(sl, device=dev)
        lg = emb[cand].double() @ hid
        best = torch.sort(lg, descending=True, stable=True)
        out.append(best.values[:k])
        prev, cur, pos = cur, int(cand[best.indices[0]]), pos + 1
        if n:
            un = w["ssm_w_in"] @ _rms64(emb[cur].double(), w["ssm_norm"], cfg["ssm_eps"])
            states.append(w["ssm_decay"] * states[-1] + (1 - w["ssm_decay"]) * un)
        hist = (hist + [code(prev, cur, states[-1] if n else None)])[-3:]
    return {"ids": None, "logits": torch.stack(out), "codes": None}


def _train64(case: dict, seed: int) -> dict:
    """Looked-up rows; the approximate surrogate's route-logit gradient; the gather's table gradients."""
    s = prepare(case, seed)
    m = s["mem"].module
    tabs = [m.tables[f"ngram_{o}"].weight.detach() for o in ORDERS]
    b, t, r = s["codes"].shape
    q, grad = s["q"].detach(), s["grad"]
    rows = torch.empty_like(grad)
    gq = torch.zeros(b, t, r, BITS, dtype=torch.float64, device="cuda")
    gt = [torch.zeros(x.shape, dtype=torch.float64, device="cuda") for x in tabs]
    for r0 in range(0, r, 8):
        c = s["codes"][:, :, r0:r0 + 8].long()
        base = torch.arange(r0, r0 + c.shape[2], device="cuda")
        for oi, (o, tab) in enumerate(zip(ORDERS, tabs)):
            cols = slice(oi * MEM, (oi + 1) * MEM)
            rows[:, :o - 1, r0:r0 + 8, cols] = 0
            nw = t - o + 1
            if nw <= 0:
                continue
            idx = base * 16 ** o + sum(c[:, k:nw + k] << (BITS * k) for k in range(o))
            rows[:, o - 1:, r0:r0 + 8, cols] = tab[idx]
            g = grad[:, o - 1:, r0:r0 + 8, cols].double()
            gt[oi].index_add_(0, idx.reshape(-1), g.reshape(-1, MEM))
            here = (tab[idx].double() * g).sum(-1)
            for e in range(o):
                for k in range(BITS):
                    flip = 1 << (BITS * e + k)
                    sign = 1.0 - 2.0 * ((idx & flip) != 0).double()
                    gq[:, e:e + nw, r0:r0 + 8, k] += ((tab[idx ^ flip].double() * g).sum(-1) - here) * sign
    p = torch.sigmoid(q.double())
    return {"rows": rows, "grad_q": gq * p * (1 - p), "grad_2": gt[0], "grad_3": gt[1]}


def _mix32(h: torch.Tensor) -> torch.Tensor:
    """MurmurHash3's 32-bit finaliser on int64 values of [0, 2^32)."""
    m = 0xFFFFFFFF
    h = h ^ (h >> 16)
    h = (h * 0x85EBCA6B) & m
    h = h ^ (h >> 13)
    h = (h * 0xC2B2AE35) & m
    return h ^ (h >> 16)


def _scaled64(case: dict, seed: int) -> torch.Tensor:
    s = prepare(case, seed)
    b, t, r = s["codes"].shape
    sl = case["scale_log2"]
    base = torch.arange(r, device="cuda")
    out = torch.zeros(b, t, MEM, dtype=torch.float64, device="cuda")
    for i in range(b):
        c = s["codes"][i].long()
        for t0 in range(0, t, 512):
            for oi, (o, tab) in enumerate(zip(ORDERS, s["tables"])):
                a, z = max(t0, o - 1), min(t, t0 + 512)
                if a >= z:
                    continue
                addr = sum(c[a - o + 1 + k:z - o + 1 + k] << (BITS * k) for k in range(o))
                p = torch.arange(i * t + a, i * t + z, device="cuda")[:, None]
                slot = _mix32(s["seed"] ^ _mix32((p * 0x9E3779B1 + base * len(ORDERS) + oi) & 0xFFFFFFFF))
                row = (((base << sl) + (slot & ((1 << sl) - 1))) << (BITS * o)) + addr
                out[i, a:z] += tab[row].double().sum(1)
    return out


@torch.no_grad()
def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("prefill", "tiny"):
        s = prepare(case, seed)
        return _layer64(s["mem"], s["h"], s["hn"])
    if kind == "sdc":
        s = prepare(case, seed)
        mem, f = s["mem"], s["mem"].router_features
        states = _scan64(s["ssm"], s["emb"])
        # the router's features are bf16 rows by definition: their rounding decides the codes' signs
        cur = _rms64(s["emb"].double(), f.cur_norm.weight.detach(), f.cur_norm.eps).to(torch.bfloat16)
        prev = torch.cat((f.start.detach().expand(s["emb"].shape[0], 1, D).to(torch.bfloat16), s["emb"][:, :-1]), 1)
        prev = _rms64(prev.double(), f.prev_norm.weight.detach(), f.prev_norm.eps).to(torch.bfloat16)
        x = torch.cat((prev, cur, states.float().to(torch.bfloat16)), -1)
        return {"states": states, "out": _layer64(mem, s["h"], x)}
    if kind in ("decode", "verify"):
        s = prepare(case, seed)
        a = max(0, case["cached"] - 11)                  # 9 conv positions, each with 2 before it
        y = _layer64(s["mem"], s["all_h"][:, a:], s["all_hn"][:, a:])
        return {"out": y[:, case["cached"] - a:], "codes": None, "conv_in": None}
    if kind == "tree_verify":
        s = prepare(case, seed)
        L, parent = case["cached"], _tree_spec(case["nodes"]).parent
        a, y = max(0, L - 11), []
        for i in range(len(parent)):
            path = [i]
            while parent[path[0]] >= 0:
                path.insert(0, parent[path[0]])
            at = list(range(a, L)) + [L + p for p in path]
            y.append(_layer64(s["mem"], s["all_h"][:, at], s["all_hn"][:, at])[:, -1])
        return {"out": torch.stack(y, 1), "codes": None, "conv_in": None}
    if kind == "draft_chain":
        return _chain64(case, seed)
    if kind == "train":
        return _train64(case, seed)
    if kind == "scaled":
        return _scaled64(case, seed)
    return None                                          # draft_tree: token ids and copied rows only
