"""Performance cases of the decode path: what a serving program does with this library, layer by layer.

Kinds of case (field "kind"):

* "append"     quantise-on-append of one layer through the cache store's `write_slots`: decode tokens (a handful per
               step, mirrored into the pinned host shadow) and prefill chunks (the mirror of a chunk runs on a stream of
               its own, bound by PCIe, and is left out: "shadow" false).
* "decode"     one decode step of `layers` layers in the one-pass form (scan, top-k, merge, blend), either replayed from
               one HIP graph ("graph" true, how a serving loop runs it) or called operator by operator.
* "two_call"   the reference-named pair of operators of one layer: Stage A (scores, top-k, statistics), then Stage B.
* "corrected"  the decode step with the CPU correction in it: one-pass form, publish to pinned memory, exact attention
               over the winners on the host's worker pool, device-side wait and blend, in one HIP graph.

Sizes are those of `jetfire_amd.workloads.CONFIGS` (32 query heads over 8 or 4 kv-heads, contexts of 4096 to 131072,
corrections of 64 to 512) and of the batches around them.  Sequence lengths of a batch are spread evenly from
"fill" * S to S ("fill" 1: all equal): a serving batch holds sequences of different ages.  Keys and values are N(0, 1)
with four key channels scaled by 8, queries N(0, 1) / sqrt(128), block tables are random permutations.
"""
from __future__ import annotations

import torch

from jetfire_amd import ops
from jetfire_amd.adapter.cache_store import JetFireInt4CacheStore

D, BLOCK = 128, 16
SCALE = D ** -0.5
CPU_THREADS = 14          # workers of the CPU correction, as bench.py

# scheme name -> key bits, value bits ("a": asymmetric keys with zero-points, "b4": INT4 keys with 64-channel groups)
BITS = {"k3v2": (3, 2), "k4v4": (4, 4), "b4v4": (4, 4), "k2v2": (2, 2), "k3v3": (3, 3), "k2v4": (2, 4), "k3v4": (3, 4),
        "a2v2": (2, 2), "a2v4": (2, 4)}


def _decode(name, B, Hq, Hkv, S, fill, scheme, group, top_k, layers, graph=True):
    return {"name": name, "kind": "decode", "B": B, "Hq": Hq, "Hkv": Hkv, "S": S, "fill": fill, "scheme": scheme,
            "group": group, "top_k": top_k, "layers": layers, "graph": graph}


def listed():
    return [
        # the append every decode step starts with: one token per running sequence, into cache and host shadow
        {"name": "append_decode_tokens", "kind": "append", "T": 5, "Hkv": 8, "scheme": "k3v2", "group": 64, "shadow": True},
        # a chunk of a prompt, ragged against the 16-token pages
        {"name": "append_prefill_chunk", "kind": "append", "T": 16371, "Hkv": 8, "scheme": "k3v2", "group": 64, "shadow": False},
        # a chat turn: one short sequence, called operator by operator (launches and host work count)
        _decode("decode_short_eager", 1, 32, 8, 777, 1.0, "k4v4", 128, 64, 1, graph=False),
        # one user at 4096 positions, a step replayed from a graph
        _decode("decode_4k_single", 1, 32, 8, 4096, 1.0, "k4v4", 128, 64, 8),
        # many short conversations at once
        _decode("decode_2k_batch32", 32, 32, 8, 2048, 0.25, "k3v2", 64, 256, 4),
        # continuous batching: sequences of very different ages under one maximum length
        _decode("decode_16k_ragged16", 16, 32, 8, 16384, 0.06, "k4v4", 128, 256, 4),
        # INT4 at the default group size (64-channel groups: the bf16 scoring model)
        _decode("decode_8k_int4_g64", 4, 32, 8, 8100, 0.5, "b4v4", 64, 256, 4),
        # eight query heads per kv-head, long contexts of different length
        _decode("decode_32k_gqa8", 4, 32, 4, 32768, 0.4, "k3v2", 64, 256, 4),
        # the headline shape: four sequences of 32768 positions
        _decode("decode_32k_batch4", 4, 32, 8, 32768, 1.0, "k3v2", 64, 256, 4),
        # one sequence of 131072 positions, INT4, wide correction
        _decode("decode_128k_single", 1, 32, 8, 131072, 1.0, "k4v4", 128, 512, 4),
        # the reference's two-operator sequence for INT4 at batch > 1
        {"name": "two_call_int4_batch4", "kind": "two_call", "B": 4, "Hq": 32, "Hkv": 8, "S": 16384, "fill": 0.5,
         "scheme": "k4v4", "group": 128, "top_k": 256},
        # end to end with the CPU correction
        {"name": "corrected_8k_batch4", "kind": "corrected", "B": 4, "Hq": 32, "Hkv": 4, "S": 8192, "fill": 0.5,
         "scheme": "k3v2", "group": 64, "top_k": 256, "layers": 2},
    ]


def _log_uniform(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def draw(rng):
    kind = rng.choices(["decode", "append", "two_call", "corrected"], [12, 4, 2, 1])[0]
    if kind == "append":
        scheme = rng.choice(["k3v2", "k3v2", "k4v4", "k2v4", "a2v2"])
        decode_tokens = rng.random() < 0.4
        T = int(_log_uniform(rng, 1, 64) if decode_tokens else _log_uniform(rng, 300, 32000))
        return {"kind": "append", "T": T, "Hkv": rng.choice([2, 4, 8]), "scheme": scheme,
                "group": rng.choice([64, 128]), "shadow": decode_tokens}
    Hkv = rng.choice([2, 4, 8, 8])
    if kind == "two_call":
        B, G = rng.randint(2, 8), rng.choice([4, 8])
        # (the score tensor of the interface bounds the context: B * Hq * S floats)
        S = int(_log_uniform(rng, 1000, 16384 * 4 * 32 / (B * G * Hkv)))
        S = min(S, 65536)
        scheme, group = rng.choice([("k4v4", 128), ("k4v4", 128), ("k3v2", 64)])
        return {"kind": "two_call", "B": B, "Hq": Hkv * G, "Hkv": Hkv, "S": S, "fill": round(rng.uniform(0.1, 1.0), 2),
                "scheme": scheme, "group": group, "top_k": rng.choice([64, 128, 256, 512])}
    if kind == "corrected":
        B, Hkv = rng.randint(1, 4), rng.choice([4, 8])
        return {"kind": "corrected", "B": B, "Hq": 32, "Hkv": Hkv, "S": int(_log_uniform(rng, 1000, 8192 * 16 / (B * Hkv))),
                "fill": round(rng.uniform(0.3, 1.0), 2), "scheme": rng.choice(["k3v2", "k4v4"]),
                "group": 128, "top_k": rng.choice([64, 128, 256]), "layers": 2}
    scheme, group = rng.choice([("k3v2", 64), ("k3v2", 64), ("k3v2", 64), ("k4v4", 128), ("k4v4", 128), ("k4v4", 128),
                                ("b4v4", 64), ("k3v2", 128), ("k2v2", 64), ("k3v3", 64), ("k2v4", 128), ("k3v4", 64),
                                ("a2v2", 128)])
    G = rng.choice([4, 4, 4, 8, 8, 1, 2, 7])
    B = int(_log_uniform(rng, 1, 33))
    # no more packed bytes per layer than the largest listed case, nor more queries than the widest one
    most = int(131072 * 8 * 132 / (B * Hkv * _row_bytes(scheme, group)) / max(1.0, G / 4))
    S = int(_log_uniform(rng, 300, min(131072, max(600, most))))
    top_k = rng.choice([64, 128, 256, 256, 512, 1024])
    while top_k > S:
        top_k //= 2
    return {"kind": "decode", "B": B, "Hq": Hkv * G, "Hkv": Hkv, "S": S,
            "fill": 1.0 if rng.random() < 0.3 else round(rng.uniform(0.05, 1.0), 2), "scheme": scheme, "group": group,
            "top_k": top_k, "layers": 4, "graph": rng.random() < 0.8}


def _row_bytes(scheme, group):
    """Packed codes and scales (zero-points) of one token of one kv-head, keys and values together."""
    kb, vb = BITS[scheme]
    return 16 * (kb + vb) + 2 * (D // group) * (3 if scheme.startswith("a") else 2)


def _lengths(case):
    B, S = case["B"], case["S"]
    low = max(1, int(S * case["fill"]))
    return [S - (S - low) * b // max(1, B - 1) for b in range(B)]


def work(case):
    if case["kind"] == "append":
        rows = case["T"] * case["Hkv"]
        return {"bytes": rows * (2 * 2 * D * (2 if case["shadow"] else 1) + _row_bytes(case["scheme"], case["group"]))
                + 8 * case["T"], "flops": rows * 2 * D * 4}
    B, Hq, Hkv, K = case["B"], case["Hq"], case["Hkv"], case["top_k"]
    tokens = sum(_lengths(case))
    packed = tokens * Hkv * _row_bytes(case["scheme"], case["group"]) + 8 * (tokens // BLOCK)
    outputs = B * Hq * (K * 16 + D * 12 + 12)          # positions and slots, o_hat, o_old, q and out, W and statistics
    if case["kind"] == "two_call":
        outputs += 2 * 4 * tokens * Hq                 # the scores, written by one operator and read by the other
    if case["kind"] == "corrected":
        outputs += B * Hq * K * 4 * D                  # the winners' bf16 rows, read by the host
    layers = case.get("layers", 1)
    return {"bytes": layers * (packed + outputs), "flops": layers * tokens * Hq * 4 * D}


def tolerance(case):
    if case["kind"] == "append":
        return "exact"
    # The same steps with the context cut into splits of 256, 512 or 1024 positions: the fp32 outputs move by at most
    # 2e-6 of their size, `out` by one bf16 step where a rounding boundary is crossed (rel 1.7e-4, max 7.7e-3 over 19
    # geometries), no winner changes.  Four times that; a score that moves by its last bit may swap at the cut.
    return {"rel": 7e-4, "max": 0.03, "differ": 1e-3}


def _cache(case, gen, slots_total):
    """One layer's packed cache in slot order, made with the library's own append, and the bf16 rows it came from."""
    Hkv, (kb, vb) = case["Hkv"], BITS[case["scheme"]]
    store = JetFireInt4CacheStore(num_kv_heads=Hkv, head_dim=D, group_size=case["group"], num_blocks=slots_total // BLOCK,
                                  block_size=BLOCK, device="cuda", k_nbits=kb, v_nbits=vb,
                                  k_asymmetric=case["scheme"].startswith("a"), shadow_enabled=False)
    k, v = _rows(slots_total, Hkv, gen)
    store.write_slots(key=k, value=v, slot_mapping=torch.arange(slots_total, device="cuda"))
    return store, k, v


def _rows(n, Hkv, gen):
    k = torch.randn(n, Hkv, D, generator=gen, device="cuda").to(torch.bfloat16)
    k[..., torch.randperm(D, generator=gen, device="cuda")[:4]] *= 8
    v = torch.randn(n, Hkv, D, generator=gen, device="cuda").to(torch.bfloat16)
    return k, v


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    if case["kind"] == "append":
        T, Hkv, (kb, vb) = case["T"], case["Hkv"], BITS[case["scheme"]]
        blocks = 2 * ((T + BLOCK - 1) // BLOCK) + 2
        store = JetFireInt4CacheStore(num_kv_heads=Hkv, head_dim=D, group_size=case["group"], num_blocks=blocks,
                                      block_size=BLOCK, device="cuda", k_nbits=kb, v_nbits=vb,
                                      k_asymmetric=case["scheme"].startswith("a"), shadow_enabled=case["shadow"])
        k, v = _rows(T, Hkv, gen)
        if case["shadow"]:        # decode tokens: one slot each, anywhere in the pool
            slots = torch.randperm(blocks * BLOCK, generator=gen, device="cuda")[:T]
        else:                     # a chunk: whole pages in any order
            pages = torch.randperm(blocks, generator=gen, device="cuda")
            slots = (pages[:, None] * BLOCK + torch.arange(BLOCK, device="cuda")).reshape(-1)[:T].contiguous()
        return {"kind": "append", "store": store, "k": k, "v": v, "slots": slots}
    B, Hq, Hkv, S, K = case["B"], case["Hq"], case["Hkv"], case["S"], case["top_k"]
    pages = (S + BLOCK - 1) // BLOCK
    lens = torch.tensor(_lengths(case), dtype=torch.int32, device="cuda")[torch.randperm(B, generator=gen, device="cuda")]
    st = {"kind": case["kind"], "case": case, "lens": lens.contiguous(), "layers": [], "graph": None,
          "table": torch.randperm(B * pages, generator=gen, device="cuda").reshape(B, pages).contiguous(),
          "q": (torch.randn(B, Hq, D, generator=gen, device="cuda") * SCALE).to(torch.bfloat16),
          "o_new": [(torch.randn(B, Hq, D, generator=gen, device="cuda") * 0.1).to(torch.bfloat16)
                    for _ in range(case.get("layers", 1))]}
    st["out"] = [torch.empty(B, Hq, D, dtype=torch.bfloat16, device="cuda") for _ in st["o_new"]]
    for _ in st["o_new"]:
        store, k, v = _cache(case, gen, B * pages * BLOCK)
        st["layers"].append(store)
        if case["kind"] == "corrected":
            ops.set_cpu_attn_threads(CPU_THREADS)
            shadow = [t.permute(1, 0, 2).contiguous().cpu() for t in (k, v)]
            st.setdefault("handoffs", []).append(ops.CpuTopkHandoff(B, Hq, Hkv, K, *shadow, SCALE))
    if case["kind"] == "corrected" or case.get("graph"):
        step = _corrected_step if case["kind"] == "corrected" else _decode_step
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            step(st)
        torch.cuda.current_stream().wait_stream(stream)
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"], stream=stream):
            st["results"] = step(st)
    return st


def _scan(st, store, **kw):
    c = st["case"]
    return ops.fused_attn_topk(c["scheme"], st["q"], store.k_data, store.k_scales, store.v_data, store.v_scales, st["table"],
                               st["lens"], c["S"], c["Hq"], c["Hkv"], BLOCK, c["top_k"], SCALE,
                               k_zp=store.k_zp if store.k_asymmetric else None, **kw)


def _decode_step(st):
    return [(_scan(st, store, blend=(o_new, out)), out) for store, o_new, out in zip(st["layers"], st["o_new"], st["out"])]


def _corrected_step(st):
    ops.pool_doorbell()
    results = []
    for store, handoff, out in zip(st["layers"], st["handoffs"], st["out"]):
        o_hat, slots, o_old, W, idx = _scan(st, store)
        handoff.stream_submit(st["q"], slots)
        handoff.stream_wait_blend(o_hat, o_old, W, out)
        results.append((o_hat, slots, o_old, W, idx, out))
    return results


def _two_call(st):
    c, store = st["case"], st["layers"][0]
    a = (st["q"], store.k_data, store.k_scales, st["table"], st["lens"], c["S"], c["Hq"], c["Hkv"], BLOCK, SCALE, c["top_k"])
    v = (store.v_data, store.v_scales, st["table"], st["lens"])
    if c["scheme"] == "k4v4":
        scores, idx, slots, m, iz = ops.int8tc_qk_scores_topk_stats(*a)
        stage_b = ops.int8tc_softmax_v_with_pre_corr_reg_stats(scores, m, iz, *v, idx, c["S"], c["Hq"], c["Hkv"], BLOCK, c["top_k"])
    else:
        scores, idx, slots = ops.int3_qk_scores_topk(*a)
        stage_b = ops.int2_softmax_v_with_pre_corr_wvs2(scores, *v, idx, c["S"], c["Hq"], c["Hkv"], BLOCK, c["top_k"])
    return [scores, idx, slots, *stage_b]


def run(state):
    if state["kind"] == "append":
        store = state["store"]
        store.write_slots(key=state["k"], value=state["v"], slot_mapping=state["slots"])
        out = [store.k_data, store.k_scales, store.v_data, store.v_scales, store.slot_filled]
        if store.k_asymmetric:
            out.append(store.k_zp)
        if store.shadow_enabled:
            out += [store.k_shadow, store.v_shadow]
        return out
    if state["graph"] is not None:
        state["graph"].replay()
        return state["results"]
    return _decode_step(state) if state["kind"] == "decode" else _two_call(state)
