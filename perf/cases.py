"""Performance cases: the calls a serving program makes around Drop + Reposition.

``listed()`` names the cases, ``draw(rng)`` gives another of the same ranges.
A case's events (dropped spans, request lengths) follow from the case itself,
so ``work`` is a function of the case; slots, K/V, queries and sinks are drawn
from the seed given to ``prepare``.

Kinds:

* ``step``     one request batch's turn end: the page-table compaction and the
               all-layer Reposition it gates (``tables.compact_rows`` +
               ``ops.reposition_kv_layers_gated``);
* ``compact``  the compaction alone, for a rank that only keeps metadata;
* ``paged``    the page-16 copy-on-write turn end (``tables.compact_pages`` +
               ``ops.reposition_kv_layers``);
* ``bind``     the slot binding of a multi-turn prompt computed in one prefill
               (``occurrence.bind_final_forward``);
* ``decode``   one decode step: read metadata from the registry rows, then
               attention of one layer of each kind the model has (full, and
               sliding-window when it has one);
* ``prefill``  one extend forward over retained prefixes: attention of one
               layer of each kind the model has.
"""

import random

import numpy as np
import torch

from akv_amd import attention, context_attention, occurrence, ops, page_table, plan, rope, synth, tables

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
LLAMA3_ROPE = dict(kind="llama3", base=500000.0, factor=8.0, original_max=8192, low_freq_factor=1.0,
                   high_freq_factor=4.0)
YARN_ROPE = dict(kind="yarn", base=150000.0, factor=32.0, original_max=4096, beta_fast=32.0, beta_slow=1.0)
PLAIN_ROPE = dict(kind="plain", base=10000.0)


def listed():
    return [
        # the smallest turn end: a 4k-token chat of a two-layer model; launches
        # and latency are all it costs
        dict(name="step-tiny-4k", kind="step", layers=2, heads=2, head_dim=64, rotary=64, dtype="bf16", neox=True,
             requests=1, n_lo=4096, n_hi=4096, spans=3, fraction=0.25, order="permutation", events=1),
        # the headline: one 32k-token GPT-OSS-120B agent request (36 layers, 8
        # KV heads x 64) drops 12 tool results on a fragmented pool
        dict(name="step-gpt-oss-32k", kind="step", layers=36, heads=8, head_dim=64, rotary=64, dtype="bf16",
             neox=True, requests=1, n_lo=32768, n_hi=32768, spans=12, fraction=0.40, order="permutation", events=2),
        # a partial-rotary fp16 model with interleaved pairs (half of a
        # 128-dim head rotates), four short ragged requests, fresh pool
        dict(name="step-partial-fp16", kind="step", layers=24, heads=4, head_dim=128, rotary=64, dtype="fp16",
             neox=False, requests=4, n_lo=1000, n_hi=8200, spans=3, fraction=0.30, order="ascending", events=3),
        # metadata of a full server: 64 requests of 2k-64k tokens compact at once
        dict(name="compact-ragged-64", kind="compact", requests=64, n_lo=2048, n_hi=65536, spans=6, fraction=0.35,
             events=3),
        # page-16 copy-on-write: four Llama-3-8B requests share an 8k system
        # prompt and each drops spans inside it
        dict(name="paged-llama3-4", kind="paged", layers=32, heads=8, head_dim=128, page=16, requests=4, prefix=8192,
             suffix_lo=1500, suffix_hi=8000, events=4),
        # slots of a 32k-token, 6-turn agent prompt computed in one prefill
        dict(name="bind-trajectory-32k", kind="bind", requests=1, n=32768, turns=6, span_lo=500, span_hi=2000,
             events=6),
        # the largest decode step: 32 GPT-OSS requests holding ~20k keys each
        # after the Drop (sinks, a full and a 128-window layer)
        dict(name="decode-gpt-oss-32x20k", kind="decode", requests=32, q_heads=64, heads=8, head_dim=64, sinks=True,
             window=128, n_lo=32768, n_hi=32768, spans=12, fraction=0.40, events=5),
        # a lightly loaded server: 4 ragged GPT-OSS requests, latency counts
        dict(name="decode-gpt-oss-4", kind="decode", requests=4, q_heads=64, heads=8, head_dim=64, sinks=True,
             window=128, n_lo=1500, n_hi=9000, spans=3, fraction=0.30, events=6),
        # Llama-3-8B (32 q / 8 KV heads x 128, full layers only), ragged batch
        dict(name="decode-llama3-12", kind="decode", requests=12, q_heads=32, heads=8, head_dim=128, sinks=False,
             window=0, n_lo=2000, n_hi=20000, spans=4, fraction=0.30, events=7),
        # a short user turn over a long retained context: 200 new tokens over
        # 19441 kept ones, a full and a 128-window GPT-OSS layer
        dict(name="prefill-turn-200", kind="prefill", q_heads=64, heads=8, head_dim=64, sinks=True, window=128,
             segments=1, new_lo=200, new_hi=200, prefix_lo=19441, prefix_hi=19441, events=8),
        # a 4096-token chunk over the same context
        dict(name="prefill-chunk-4096", kind="prefill", q_heads=64, heads=8, head_dim=64, sinks=True, window=128,
             segments=1, new_lo=4096, new_hi=4096, prefix_lo=19441, prefix_hi=19441, events=9),
        # mixed turns of a Llama-3-8B batch: 6 ragged segments over ragged prefixes
        dict(name="prefill-llama3-6", kind="prefill", q_heads=32, heads=8, head_dim=128, sinks=False, window=0,
             segments=6, new_lo=33, new_hi=900, prefix_lo=700, prefix_hi=16000, events=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(("step", "step", "compact", "paged", "bind", "decode", "decode", "prefill", "prefill"))
    c = dict(kind=kind, events=rng.randrange(1 << 20))
    if kind == "step":
        head_dim = rng.choice((64, 128))
        requests = rng.randint(1, 4)
        c.update(layers=_log_int(rng, 2, 36), heads=rng.choice((2, 4, 8)), head_dim=head_dim,
                 rotary=rng.choice((head_dim, head_dim, head_dim // 2)), dtype=rng.choice(("bf16", "bf16", "fp16", "fp32")),
                 neox=rng.random() < 0.7, requests=requests, spans=rng.randint(1, 12),
                 fraction=round(rng.uniform(0.1, 0.5), 3), order=rng.choice(("permutation", "ascending")))
        c["n_hi"] = _log_int(rng, 1000, 32768 // requests)
        c["n_lo"] = max(700, c["n_hi"] // rng.randint(1, 4))
        c["n_hi"] = max(c["n_hi"], c["n_lo"])
        # no larger than the headline's pool
        row = 2 * c["heads"] * head_dim * DTYPES[c["dtype"]].itemsize
        most = 36 * 65537 * 2 * 8 * 64 * 2
        c["layers"] = max(1, min(c["layers"], most // (row * 2 * c["n_hi"] * requests)))
    elif kind == "compact":
        hi = _log_int(rng, 2000, 65536)
        c.update(requests=_log_int(rng, 8, 64), n_lo=max(600, hi // rng.randint(1, 32)), n_hi=hi,
                 spans=rng.randint(1, 8), fraction=round(rng.uniform(0.1, 0.6), 3))
    elif kind == "paged":
        hi = _log_int(rng, 500, 8000)
        c.update(layers=_log_int(rng, 4, 32), heads=8, head_dim=128, page=16, requests=rng.randint(2, 4),
                 prefix=16 * _log_int(rng, 64, 512), suffix_lo=max(100, hi // 4), suffix_hi=hi)
    elif kind == "bind":
        c.update(requests=rng.randint(1, 3), n=_log_int(rng, 3000, 32768), turns=rng.randint(3, 8),
                 span_lo=20, span_hi=rng.randint(100, 2000))
    elif kind == "decode":
        gpt = rng.random() < 0.6
        requests = _log_int(rng, 1, 32)
        hi = _log_int(rng, 300, 32768)
        c.update(requests=requests, q_heads=64 if gpt else 32, heads=8, head_dim=64 if gpt else 128, sinks=gpt,
                 window=128 if gpt else 0, n_lo=max(200, hi // rng.randint(1, 6)), n_hi=hi, spans=rng.randint(1, 8),
                 fraction=round(rng.uniform(0.1, 0.5), 3))
    else:
        gpt = rng.random() < 0.6
        segments = rng.randint(1, 6)
        new = _log_int(rng, 16, 4096 // segments)
        prefix = _log_int(rng, 300, 19441)
        c.update(q_heads=64 if gpt else 32, heads=8, head_dim=64 if gpt else 128, sinks=gpt, window=128 if gpt else 0,
                 segments=segments, new_lo=max(1, new // rng.randint(1, 8)), new_hi=new,
                 prefix_lo=max(100, prefix // rng.randint(1, 8)), prefix_hi=prefix)
    return c


# ---------------------------------------------------------------------------
# What follows from the case alone: lengths, dropped spans, layouts.


def _lengths(c, rng, count, lo, hi):
    return [rng.randint(c[lo], c[hi]) for _ in range(count)]


def _spans(c, rng, n):
    """Dropped spans of one request: ``spans`` seeded spans of ``fraction`` of it."""
    k = max(1, min(c["spans"], n // 64))
    g = np.random.default_rng(rng.randrange(1 << 31))
    total = max(k, int(c["fraction"] * n))
    return synth.place_spans(g, n, synth.split_total(g, total, k))


def _requests(c):
    rng = random.Random(c["events"])
    ns = _lengths(c, rng, c["requests"], "n_lo", "n_hi")
    return ns, [_spans(c, rng, n) for n in ns]


def _layouts(c):
    ns, spans = _requests(c)
    return ns, [plan.compile_context_layout(**synth.request_events(n, s)) for n, s in zip(ns, spans)]


def _counts(ns, spans):
    """(kept, moved) of each request: a closing Reposition moves every kept
    token behind the first dropped one."""
    kept = [n - sum(e - s for s, e in sp) for n, sp in zip(ns, spans)]
    return kept, [k - sp[0][0] for k, sp in zip(kept, spans)]


def _paged_workload(c):
    m = synth.Model("paged", c["layers"], c["heads"], c["head_dim"], c["head_dim"], LLAMA3_ROPE)
    return synth.shared_prefix_workload("paged", m, c["requests"], c["prefix"], c["suffix_lo"], c["suffix_hi"], 1, 3,
                                        min(64, c["prefix"] // 16), min(512, c["prefix"] // 8), c["page"],
                                        c["events"])


def _trajectories(c):
    rng = random.Random(c["events"])
    out = []
    for _ in range(c["requests"]):
        events, visible = synth.trajectory_events(c["n"], c["turns"], c["span_lo"], c["span_hi"],
                                                  rng.randrange(1 << 20))
        lay = plan.compile_context_layout(**events)
        out.append((lay, occurrence.compile_occurrence_window(lay, visible, lay.positions, query_start=0,
                                                               query_end=c["n"])))
    return out


def _segments(c):
    rng = random.Random(c["events"])
    return (_lengths(c, rng, c["segments"], "new_lo", "new_hi"),
            _lengths(c, rng, c["segments"], "prefix_lo", "prefix_hi"))


# ---------------------------------------------------------------------------
# Inputs.


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _slots(order, first, total, seed):
    """``total`` distinct slots from ``first`` on: the free list of a
    fragmented or of a fresh pool."""
    if order == "ascending":
        return np.arange(first, first + total, dtype=np.int32)
    return (np.random.default_rng(seed).permutation(total) + first).astype(np.int32)


def _pool(shape, dtype, gen):
    """K and V of all layers [layers, slots, heads, dim] and their per-layer addresses."""
    kv = [torch.randn(shape, generator=gen, device="cuda", dtype=dtype) for _ in range(2)]
    ptrs = [torch.tensor([t[l].data_ptr() for l in range(shape[0])], dtype=torch.uint64).to("cuda") for t in kv]
    return kv[0], kv[1], ptrs[0], ptrs[1]


def _rope_table(spec, dim, positions):
    spec = dict(spec)
    return rope.make_table(spec.pop("kind"), dim, positions, dtype=torch.float32, device="cuda", **spec)


def _prepare_compaction(c, seed, order):
    ns, layouts = _layouts(c)
    spans = _requests(c)[1]
    kept, moved = _counts(ns, spans)
    total = sum(ns) + sum(moved) + len(ns)
    free = _slots(order, 1, total, seed)
    birth, fresh = free[: sum(ns)], free[sum(ns): sum(ns) + sum(moved)]
    table = torch.full((len(ns) + 1, max(ns) + 8), -1, dtype=torch.int32)
    for b, n in enumerate(ns):  # one generated token after each prompt
        table[b + 1, n] = int(free[sum(ns) + sum(moved) + b])
    inputs = tables.pack_compaction_inputs(layouts, "cuda")
    return dict(
        inputs=inputs, out=tables.allocate_outputs(inputs, "cuda", generated_total=len(ns)), table=table.to("cuda"),
        rows=torch.arange(1, len(ns) + 1, dtype=torch.int64, device="cuda"), fresh=torch.from_numpy(fresh).to("cuda"),
        birth=torch.from_numpy(birth).to("cuda"), generated=torch.ones(len(ns), dtype=torch.int32, device="cuda"),
        slots=total + 1, positions=max(ns),
    )


def _prepare_paged(c, seed):
    w = _paged_workload(c)
    w = synth.replace(w, seed=seed)  # page ids are the seed's, the events the case's
    a = synth.assign_pages(w)
    layouts = synth.compile_layouts(w)
    inputs = tables.pack_paged_inputs(layouts, c["page"], "cuda")
    k, v, kp, vp = _pool((c["layers"], a.pool_pages * c["page"], c["heads"], c["head_dim"]), torch.bfloat16, _gen(seed))
    return dict(
        inputs=inputs, out=tables.allocate_paged_outputs(inputs, "cuda"),
        table=torch.full((c["requests"], max(w.lengths) + 8), -1, dtype=torch.int32, device="cuda"),
        rows=torch.arange(c["requests"], dtype=torch.int64, device="cuda"),
        fresh=torch.from_numpy(np.concatenate(a.fresh_pages)).to("cuda"),
        birth=torch.from_numpy(np.concatenate(a.birth_rows)).to("cuda"),
        k=k, v=v, k_ptrs=kp, v_ptrs=vp, rope=_rope_table(LLAMA3_ROPE, c["head_dim"], max(w.lengths)),
    )


def _prepare_bind(c, seed):
    got = _trajectories(c)
    inputs = occurrence.pack_final_forward([w for _, w in got], [np.asarray(l.keep_mask, dtype=bool) for l, _ in got],
                                           "cuda")
    n, extra = sum(inputs.n_tokens), sum(inputs.extra)
    free = _slots("permutation", 1, n + extra, seed)
    return dict(
        inputs=inputs, out=occurrence.allocate_final_forward_outputs(inputs, "cuda"),
        table=torch.full((c["requests"], c["n"] + 8), -1, dtype=torch.int32, device="cuda"),
        rows=torch.arange(c["requests"], dtype=torch.int64, device="cuda"),
        birth=torch.from_numpy(free[:n]).to("cuda"), fresh=torch.from_numpy(free[n:]).to("cuda"),
    )


def _prepare_decode(c, seed):
    ns, spans = _requests(c)
    kept, moved = _counts(ns, spans)
    B, width = len(ns), max(ns) + 8
    gen = _gen(seed)
    slots = sum(ns) + sum(moved) + B + 1
    free = _slots("permutation", 1, slots - 1, seed)
    table = np.full((B, width), -1, dtype=np.int32)
    raw_ids, at = [], 0
    for b, (n, sp) in enumerate(zip(ns, spans)):
        keep = np.ones(n, dtype=bool)
        for s, e in sp:
            keep[s:e] = False
        raw = np.flatnonzero(keep).astype(np.int32)
        table[b, raw] = free[at: at + len(raw)]
        table[b, n] = free[at + len(raw)]  # the token being decoded
        at += len(raw) + 1
        raw_ids.append(raw)
    raw_dev = torch.from_numpy(np.concatenate(raw_ids)).to("cuda")
    pos_dev = torch.from_numpy(np.concatenate([np.arange(k, dtype=np.int32) for k in kept])).to("cuda")
    off = np.concatenate(([0], np.cumsum(kept)))
    registry = torch.tensor([(raw_dev.data_ptr() + 4 * int(off[b]), pos_dev.data_ptr() + 4 * int(off[b]), ns[b],
                              kept[b], kept[b], 0) for b in range(B)], dtype=torch.int64).to("cuda")
    heads, d = c["heads"], c["head_dim"]
    max_len = max(kept) + 1
    s = dict(
        registry=registry, keep_alive=(raw_dev, pos_dev), table=torch.from_numpy(table).to("cuda"),
        rows=torch.arange(B, dtype=torch.int64, device="cuda"),
        seq=torch.tensor([k + 1 for k in kept], dtype=torch.int64, device="cuda"),
        indptr=torch.zeros(B + 1, dtype=torch.int32, device="cuda"),
        indices=torch.zeros(sum(kept) + B, dtype=torch.int32, device="cuda"),
        q=torch.randn((B, c["q_heads"], d), generator=gen, device="cuda", dtype=torch.bfloat16),
        k=torch.randn((slots, heads, d), generator=gen, device="cuda", dtype=torch.bfloat16),
        v=torch.randn((slots, heads, d), generator=gen, device="cuda", dtype=torch.bfloat16),
        sinks=torch.randn(c["q_heads"], generator=gen, device="cuda") if c["sinks"] else None,
        out=torch.empty((B, c["q_heads"], d), dtype=torch.bfloat16, device="cuda"), max_len=max_len,
        workspace=torch.empty(attention.workspace_bytes(B, heads, d, max_len) // 4 + 1, dtype=torch.float32,
                              device="cuda"),
        lengths=[k + 1 for k in kept],
        active=[np.concatenate((table[b, raw], table[b, ns[b]: ns[b] + 1])) for b, raw in enumerate(raw_ids)],
        window=c["window"],
    )
    if c["window"]:
        s.update(win_len=torch.empty_like(s["seq"]), win_start=torch.empty_like(s["seq"]),
                 win_indptr=torch.zeros(B + 1, dtype=torch.int32, device="cuda"),
                 win_indices=torch.zeros(B * (c["window"] + 1), dtype=torch.int32, device="cuda"),
                 win_out=torch.empty_like(s["out"]))
    return s


def _prepare_prefill(c, seed):
    new, prefix = _segments(c)
    gen = _gen(seed)
    total, keys = sum(new), sum(prefix)
    slots = 2 * keys + 1
    heads, d = c["heads"], c["head_dim"]

    def randn(*shape):
        return torch.randn(shape, generator=gen, device="cuda", dtype=torch.bfloat16)

    qpos, kpos = [], []
    for m, p in zip(new, prefix):  # a dropped span not yet repositioned leaves a hole
        at = np.arange(p + m, dtype=np.int64)
        at[p // 2:] += p // 8
        kpos.append(at[:p])
        qpos.append(at[p:])
    q = randn(total, c["q_heads"], d)
    return dict(
        q=q, k=randn(total, heads, d), v=randn(total, heads, d), k_pool=randn(slots, heads, d),
        v_pool=randn(slots, heads, d),
        indices=torch.from_numpy(_slots("permutation", 1, slots - 1, seed)[:keys].copy()).to("cuda"),
        qo=torch.from_numpy(np.concatenate(([0], np.cumsum(new)))).to("cuda"),
        kv=torch.from_numpy(np.concatenate(([0], np.cumsum(prefix)))).to("cuda"),
        q_pos=torch.from_numpy(np.concatenate(qpos)).to("cuda"), k_pos=torch.from_numpy(np.concatenate(kpos)).to("cuda"),
        sinks=torch.randn(c["q_heads"], generator=gen, device="cuda") if c["sinks"] else None,
        out=torch.empty_like(q), win_out=torch.empty_like(q) if c["window"] else None, window=c["window"],
        longest=max(new), scale=d ** -0.5,
    )


def prepare(case, seed):
    kind = case["kind"]
    if kind == "compact":
        s = _prepare_compaction(case, seed, "permutation")
    elif kind == "step":
        s = _prepare_compaction(case, seed, case["order"])
        s["k"], s["v"], s["k_ptrs"], s["v_ptrs"] = _pool(
            (case["layers"], s["slots"], case["heads"], case["head_dim"]), DTYPES[case["dtype"]], _gen(seed))
        s["rope"] = _rope_table(_step_rope(case), case["rotary"], s["positions"])
        s["neox"], s["rotary"] = case["neox"], case["rotary"]
    elif kind == "paged":
        s = _prepare_paged(case, seed)
    elif kind == "bind":
        s = _prepare_bind(case, seed)
    elif kind == "decode":
        s = _prepare_decode(case, seed)
    else:
        s = _prepare_prefill(case, seed)
    s["kind"] = kind
    return s


def _step_rope(c):
    return YARN_ROPE if c["layers"] == 36 else PLAIN_ROPE


# ---------------------------------------------------------------------------
# One pass.


def _compaction_outputs(s):
    o = s["out"]
    return dict(table=s["table"], retired=o.retired, copy_src=o.copy_src, copy_dst=o.copy_dst, copy_pairs=o.copy_pairs,
                raw_indices=o.raw_indices, active_positions=o.active_positions, kv_indices=o.kv_indices,
                kv_indptr=o.kv_indptr, last_page_len=o.last_page_len, counts=o.counts)


def run(s):
    kind, o = s["kind"], s.get("out")
    if kind in ("compact", "step"):
        tables.compact_rows(s["inputs"], s["table"], s["rows"], s["fresh"], o, generated=s["generated"],
                            birth_slots=s["birth"])
        if kind == "compact":
            return _compaction_outputs(s)
        ops.reposition_kv_layers_gated(s["k_ptrs"], s["v_ptrs"], s["k"][0], s["v"][0], o.copy_src, o.copy_dst,
                                       o.copy_pairs, s["rope"], status=o.status, is_neox_style=s["neox"],
                                       rotary_dim=s["rotary"])
        return dict(_compaction_outputs(s), k=s["k"], v=s["v"])
    if kind == "paged":
        tables.compact_pages(s["inputs"], s["table"], s["rows"], s["fresh"], o, birth_slots=s["birth"])
        ops.reposition_kv_layers(s["k_ptrs"], s["v_ptrs"], s["k"][0], s["v"][0], o.copy_src, o.copy_dst, o.copy_pairs,
                                 s["rope"])
        return dict(table=s["table"], copy_src=o.copy_src, copy_dst=o.copy_dst, copy_pairs=o.copy_pairs,
                    released=o.released_pages, page_table=o.page_table, raw_indices=o.raw_indices,
                    active_positions=o.active_positions, k=s["k"], v=s["v"])
    if kind == "bind":
        occurrence.bind_final_forward(s["inputs"], s["table"], s["rows"], s["birth"], s["fresh"], o)
        return dict(table=s["table"], slots=o.occurrence_slots, copy_src=o.copy_src, copy_dst=o.copy_dst,
                    copy_pairs=o.copy_pairs, retired=o.retired)
    if kind == "decode":
        scale = s["q"].shape[-1] ** -0.5
        page_table.build_indptr(s["seq"], s["indptr"])
        page_table.context_decode_indices(s["registry"], s["table"], s["rows"], s["seq"], s["indptr"], s["indices"])
        attention.decode_attention(s["q"], s["k"], s["v"], s["indptr"], s["indices"], o, scale=scale,
                                   max_len=s["max_len"], sinks=s["sinks"], workspace=s["workspace"])
        got = dict(indptr=s["indptr"], indices=s["indices"], out=o)
        if s["window"]:
            page_table.context_window_lengths(s["registry"], s["rows"], s["seq"], s["win_len"], s["window"],
                                              starts=s["win_start"])
            page_table.build_indptr(s["win_len"], s["win_indptr"])
            page_table.context_decode_indices(s["registry"], s["table"], s["rows"], s["win_len"], s["win_indptr"],
                                              s["win_indices"], starts=s["win_start"])
            attention.decode_attention(s["q"], s["k"], s["v"], s["win_indptr"], s["win_indices"], s["win_out"],
                                       scale=scale, max_len=s["window"] + 1, sinks=s["sinks"],
                                       workspace=s["workspace"])
            got.update(win_indptr=s["win_indptr"], win_indices=s["win_indices"], win_out=s["win_out"])
        return got
    got = {}
    for name, window in (("out", -1), ("win_out", s["window"])):
        if s[name] is None:
            continue
        got[name] = context_attention.extend_attention_fwd(
            s["q"], s["k"], s["v"], s[name], s["k_pool"], s["v_pool"], s["qo"], s["kv"], s["indices"], None, True,
            None, s["longest"], sm_scale=s["scale"], sliding_window_size=window, sinks=s["sinks"],
            context_q_positions=s["q_pos"], context_kv_positions=s["k_pos"])
    return got


# ---------------------------------------------------------------------------
# What a pass cannot do without.


def work(case):
    c, kind = case, case["kind"]
    if kind in ("compact", "step"):
        ns, spans = _requests(c)
        kept, moved = (sum(x) for x in _counts(ns, spans))
        n = sum(ns)
        retired = n - kept + moved
        # keep, birth and final positions, birth slots in; rows and lists out
        size = n * (1 + 4 + 4 + 4 + 4) + 4 * moved + 4 * retired + 16 * moved + 12 * kept
        flops = 0
        if kind == "step":
            e = DTYPES[c["dtype"]].itemsize
            size += moved * (4 * c["layers"] * c["heads"] * c["head_dim"] * e + 16 + 8 * c["rotary"])
            flops = moved * c["layers"] * c["heads"] * c["rotary"] // 2 * 14
        return dict(bytes=size, flops=flops)
    if kind == "paged":
        w = _paged_workload(c)
        copies = sum(kept - p0 * c["page"] for kept, p0, _ in synth.paged_demand(w))
        kept = sum(d[0] for d in synth.paged_demand(w))
        size = sum(w.lengths) * 17 + copies * 16 + kept * 8
        size += copies * (4 * c["layers"] * c["heads"] * c["head_dim"] * 2 + 16 + 8 * c["head_dim"])
        return dict(bytes=size, flops=copies * c["layers"] * c["heads"] * c["head_dim"] // 2 * 14)
    if kind == "bind":
        got = _trajectories(c)
        occ, n = sum(w.occurrence_count for _, w in got), c["requests"] * c["n"]
        copies = occ - n
        # occurrence raw and position, terminal occurrence, keep, birth slot in;
        # occurrence slots, rows, copy lists, retired slots out
        return dict(bytes=8 * occ + 9 * n + 4 * copies + 4 * occ + 4 * n + 16 * copies + 4 * copies, flops=0)
    if kind == "decode":
        ns, spans = _requests(c)
        keys = [k + 1 for k in _counts(ns, spans)[0]]
        read = [keys] + ([[min(k, c["window"] + 1) for k in keys]] if c["window"] else [])
        total = sum(sum(r) for r in read)
        size = total * (2 * 2 * c["heads"] * c["head_dim"] + 12)
        size += len(read) * 2 * 2 * c["requests"] * c["q_heads"] * c["head_dim"]
        return dict(bytes=size, flops=4 * total * c["q_heads"] * c["head_dim"])
    new, prefix = _segments(c)
    q, kv = sum(new) * c["q_heads"] * c["head_dim"] * 2, c["heads"] * c["head_dim"] * 2
    size = 2 * q + (sum(new) + sum(prefix)) * 2 * kv + sum(prefix) * 12 + sum(new) * 8
    pairs = sum(m * p + m * (m + 1) // 2 for m, p in zip(new, prefix))
    if c["window"]:
        W = c["window"]
        size += 2 * q + sum(m + min(p, W) for m, p in zip(new, prefix)) * 2 * kv
        pairs += sum(min(p + i + 1, W + 1) for m, p in zip(new, prefix) for i in range(m))
    return dict(bytes=size, flops=4 * pairs * c["q_heads"] * c["head_dim"])


def tolerance(case):
    # positions, slots and moved K/V are bit for bit the reference's; attention
    # rounds its weights and its output to bf16 (measured 2.1e-3 to 2.4e-3 from
    # the 64-bit result)
    if case["kind"] in ("decode", "prefill"):
        return {"rel": 0.009, "max": 0.06}
    return "exact"


# ---------------------------------------------------------------------------
# The same outputs in 64 bits.


def _exact_reposition(s, src, dst, pairs, rotary, neox):
    """K and V after the moves, float64: inverse rotation from the old
    position, then rotation to the new one."""
    k, v = s["k"].double(), s["v"].double()
    half = rotary // 2
    src, dst = (torch.as_tensor(x, dtype=torch.int64, device="cuda") for x in (src, dst))
    old, new = (torch.as_tensor(pairs[:, i].copy(), dtype=torch.int64, device="cuda") for i in (0, 1))
    t = s["rope"].double()
    co, so, cn, sn = (x[:, None, :] for x in (t[old, :half], t[old, half:], t[new, :half], t[new, half:]))
    norm = co * co + so * so
    for l in range(k.shape[0]):
        x = k[l][src]
        a, b = (x[..., :half], x[..., half:rotary]) if neox else (x[..., 0:rotary:2], x[..., 1:rotary:2])
        u, w = (a * co + b * so) / norm, (b * co - a * so) / norm
        a, b = u * cn - w * sn, w * cn + u * sn
        y = x.clone()
        if neox:
            y[..., :half], y[..., half:rotary] = a, b
        else:
            y[..., 0:rotary:2], y[..., 1:rotary:2] = a, b
        k[l][dst] = y
        v[l][dst] = v[l][src]
    return k, v


def _exact_attention(q, keys, values, sinks, scale, visible):
    """One q-head group: q [n, G, D], keys/values [m, D], visible [n, m] or None."""
    s = torch.matmul(q.reshape(-1, q.shape[-1]), keys.t().contiguous()).view(q.shape[0], q.shape[1], -1) * scale
    if visible is not None:
        s = s.masked_fill(~visible[:, None, :], float("-inf"))
    top = s.amax(-1, keepdim=True)
    if sinks is not None:
        top = torch.maximum(top, sinks.view(1, -1, 1))
    p = torch.exp(s - top)
    norm = p.sum(-1, keepdim=True)
    if sinks is not None:
        norm = norm + torch.exp(sinks.view(1, -1, 1) - top)
    return torch.matmul((p / norm).view(-1, p.shape[-1]), values).view(q.shape)


def _exact_decode(s, window):
    q = s["q"].double()
    out = torch.empty_like(q)
    heads = s["k"].shape[1]
    group = q.shape[1] // heads
    for b, slots in enumerate(s["active"]):
        slots = torch.from_numpy(np.asarray(slots[-(window + 1):] if window else slots, dtype=np.int64)).to("cuda")
        k, v = s["k"][slots].double(), s["v"][slots].double()
        for h in range(heads):
            g = slice(h * group, (h + 1) * group)
            sinks = s["sinks"][g].double() if s["sinks"] is not None else None
            out[b: b + 1, g] = _exact_attention(q[b: b + 1, g], k[:, h].contiguous(), v[:, h].contiguous(), sinks,
                                                q.shape[-1] ** -0.5, None)
    return out


def _exact_prefill(s, window):
    out = torch.empty_like(s["q"], dtype=torch.float64)
    heads = s["k"].shape[1]
    group = s["q"].shape[1] // heads
    qo, kv = s["qo"].tolist(), s["kv"].tolist()
    for i in range(len(qo) - 1):
        q0, q1 = qo[i], qo[i + 1]
        idx = s["indices"][kv[i]: kv[i + 1]].long()
        kpos = torch.cat((s["k_pos"][kv[i]: kv[i + 1]], s["q_pos"][q0:q1]))
        p = len(idx)
        for h in range(heads):
            g = slice(h * group, (h + 1) * group)
            k = torch.cat((s["k_pool"][idx, h], s["k"][q0:q1, h])).double()
            v = torch.cat((s["v_pool"][idx, h], s["v"][q0:q1, h])).double()
            sinks = s["sinks"][g].double() if s["sinks"] is not None else None
            for a in range(q0, q1, 512):
                e = min(a + 512, q1)
                at = torch.arange(a - q0, e - q0, device="cuda")
                see = torch.arange(p + q1 - q0, device="cuda")[None, :] <= (at + p)[:, None]
                if window:
                    see &= s["q_pos"][a:e, None] <= kpos[None, :] + window
                out[a:e, g] = _exact_attention(s["q"][a:e, g].double(), k, v, sinks, s["scale"], see)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("compact", "bind"):
        return None  # whole numbers only
    s = prepare(case, seed)
    if kind == "step":
        ns, layouts = _layouts(case)
        birth, fresh = s["birth"].cpu().numpy(), s["fresh"].cpu().numpy()
        old = np.concatenate([np.asarray(l.birth_positions) for l in layouts])
        new = np.concatenate([np.asarray(l.positions) for l in layouts])
        moved = np.concatenate([np.asarray(l.keep_mask) for l in layouts]) & (old != new)
        k, v = _exact_reposition(s, birth[moved], fresh, np.stack((old[moved], new[moved]), 1), case["rotary"],
                                 case["neox"])
        return dict(k=k, v=v)
    if kind == "paged":
        w = _paged_workload(case)
        birth, fresh = s["birth"].cpu().numpy(), s["fresh"].cpu().numpy()
        at = got = 0
        src, dst, pairs = [], [], []
        for n, lay, (kept, p0, pages) in zip(w.lengths, synth.compile_layouts(w), synth.paged_demand(w)):
            raw = np.flatnonzero(np.asarray(lay.keep_mask))[p0 * case["page"]:]
            rank = np.arange(p0 * case["page"], kept)
            src.append(birth[at + raw])
            dst.append(fresh[got + rank // case["page"] - p0] * case["page"] + rank % case["page"])
            pairs.append(np.stack((np.asarray(lay.birth_positions)[raw], rank), 1))
            at, got = at + n, got + pages
        k, v = _exact_reposition(s, *(np.concatenate(x) for x in (src, dst, pairs)), case["head_dim"], True)
        return dict(k=k, v=v)
    of = _exact_decode if kind == "decode" else _exact_prefill
    return dict(out=of(s, 0), **({"win_out": of(s, case["window"])} if case["window"] else {}))
