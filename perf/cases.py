"""The calls whose speed is measured, with inputs, exact results and tolerances.

Every case drives the C entry points through the ctypes binding the way a
serving program does: buffers, tables and workspaces are made once, the
launches of a step are captured into a HIP graph (as bench.py and the graph
tests do) and a pass replays it.  Four kinds:

* ``decode``  one decode step over ``layers`` layers: the fp16 append (or RoPE)
  and the attention of every session.  ``form`` is the call used: ``planned``
  (plan once, launch_attn_decode_paged_planned per layer), ``rope`` (the same
  with RopeKvOp fused), ``rope_solo`` (one launch per layer, short contexts) or
  ``calls`` (the reference's signatures: launch_rope_kv_store_paged and
  launch_attn_decode_paged per layer and session).
* ``prefill`` one chunk of ``n_q`` tokens per session: RoPE + append, then
  causal attention.  ``form`` is ``batch`` or ``calls`` (one session per call).
* ``gemv``    the Q4_K projections of ``layers`` decode layers, for one token
  (launch_gemv_q4k_f32, launch_quant_q8, launch_gemv_q4k) or for four
  (launch_quant_q8, launch_gemv4_q4k).
* ``cow``     the page copies of a batch of forked sessions' first append.

Contexts are drawn from [ctx_lo, ctx_hi] (prefixes from [past_lo, past_hi]) with
the case's own ``mix``, so every seed does the same amount of work; pages are
scattered over the pool by a seeded shuffle.
"""
import ctypes
import math
import sys
import weakref
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "conflux-nova_amd"))
import nova_amd  # noqa: E402

KB = 16                      # tokens per page
HD = 128
HALF = HD // 2
# query heads, kv heads, layers
MODELS = {"qwen25_1p5b": (12, 2, 28), "qwen25_7b": (28, 4, 28), "qwen25_14b": (40, 8, 48)}
# hidden, key/value and FFN widths of their projections
_WIDTHS = {"qwen25_1p5b": (1536, 256, 8960), "qwen25_7b": (3584, 512, 18944), "qwen25_14b": (5120, 1024, 13824)}
THETA = 1e6


def listed():
    return [
        # one user, the small model, a chat of 1024 tokens: latency and launches
        dict(name="decode_1p5b_single", kind="decode", form="planned", model="qwen25_1p5b", sessions=1, ctx_lo=1024,
             ctx_hi=1024, mix=1, layers=28),
        # the benchmark's own step: a ragged batch of 16 sessions
        dict(name="decode_7b_ragged16", kind="decode", form="planned", model="qwen25_7b", sessions=16, ctx_lo=512,
             ctx_hi=8192, mix=2024, layers=28),
        # long documents on the large model (the benchmark's 8 x 32768, 4 of its 48 layers)
        dict(name="decode_14b_long", kind="decode", form="planned", model="qwen25_14b", sessions=8, ctx_lo=32768,
             ctx_hi=32768, mix=1, layers=4),
        # many short chats at once, RoPE fused, one launch per layer
        dict(name="decode_7b_short_chats", kind="decode", form="rope_solo", model="qwen25_7b", sessions=24, ctx_lo=17,
             ctx_hi=600, mix=7, layers=28),
        # the reference's own decode loop: one session, one call per op and layer
        dict(name="decode_7b_calls", kind="decode", form="calls", model="qwen25_7b", sessions=1, ctx_lo=2047,
             ctx_hi=2047, mix=1, layers=28),
        # the benchmark's chunked prefill: 8 sessions x 512 tokens over ragged prefixes
        dict(name="prefill_7b_batch", kind="prefill", form="batch", model="qwen25_7b", sessions=8, n_q=512, past_lo=0,
             past_hi=4096, mix=2024, layers=2),
        # one session's chunk in the middle of a prompt, the reference's signature
        dict(name="prefill_7b_chunk", kind="prefill", form="calls", model="qwen25_7b", sessions=1, n_q=512,
             past_lo=1536, past_hi=1536, mix=1, layers=4),
        # a first short prompt on the small model
        dict(name="prefill_1p5b_prompt", kind="prefill", form="calls", model="qwen25_1p5b", sessions=1, n_q=173,
             past_lo=0, past_hi=0, mix=1, layers=28),
        # a follow-up question behind a long document on the large model
        dict(name="prefill_14b_followup", kind="prefill", form="calls", model="qwen25_14b", sessions=1, n_q=300,
             past_lo=12001, past_hi=12001, mix=1, layers=2),
        # the projections of one token
        dict(name="gemv_7b_token", kind="gemv", model="qwen25_7b", tokens=1, hidden=3584, kv=512, ffn=18944, layers=2),
        # the projections of a decode batch of four
        dict(name="gemv_7b_four", kind="gemv", model="qwen25_7b", tokens=4, hidden=3584, kv=512, ffn=18944, layers=2),
        # 64 sessions forked from 4 prompts write their first token
        dict(name="cow_7b_fork", kind="cow", model="qwen25_7b", children=64, donors=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: any model, sizes spread over their logarithm."""
    model = rng.choice(sorted(MODELS))
    nh, nkv, n_layers = MODELS[model]
    kind = rng.choice(["decode"] * 5 + ["prefill"] * 4 + ["gemv"] * 2 + ["cow"])
    mix = rng.randrange(1 << 20)
    if kind == "decode":
        form = rng.choice(["planned", "planned", "rope", "rope_solo", "calls"])
        hi = _log(rng, 17, {"rope_solo": 640, "calls": 8192}.get(form, 32768))
        lo = rng.randint(max(1, hi // 16), hi)
        sessions = _log(rng, 1, 4 if form == "calls" else 32)
        # the pools stay under 2.5 GB, the largest listed case's under 4.4 GB
        while sessions > 1 and sessions * hi * nkv * HD * 4 > 2.5e9:
            sessions -= 1
        layers = max(1, min(n_layers, int(2.5e9 // (sessions * hi * nkv * HD * 4))))
        return dict(kind="decode", form=form, model=model, sessions=sessions, ctx_lo=lo, ctx_hi=hi, mix=mix,
                    layers=layers)
    if kind == "prefill":
        form = rng.choice(["batch", "calls"])
        n_q = _log(rng, 16, 1024)
        hi = _log(rng, 1, 16384)
        lo = rng.choice([0, rng.randint(0, hi), hi])
        sessions = _log(rng, 1, 8) if form == "batch" else _log(rng, 1, 2)

        def flops():
            return sessions * n_q * nh * 4.0 * HD * (hi + n_q)

        while sessions > 1 and flops() > 1.5e11:
            sessions -= 1
        layers = max(1, min(n_layers, int(2.0e11 // flops())))
        return dict(kind="prefill", form=form, model=model, sessions=sessions, n_q=n_q, past_lo=lo, past_hi=hi,
                    mix=mix, layers=layers)
    if kind == "gemv":
        # a model's own widths, or any others in whole super-blocks of 256
        hidden, kv, ffn = _WIDTHS[model] if rng.random() < 0.4 else (
            256 * _log(rng, 4, 24), 128 * rng.randint(1, 10), 256 * _log(rng, 8, 80))
        per = (2 * hidden * (hidden + kv) + 3 * hidden * ffn) * 144 // 256
        return dict(kind="gemv", model=model, tokens=rng.choice([1, 4]), hidden=hidden, kv=kv, ffn=ffn,
                    layers=max(1, min(rng.randint(1, 12), int(3.5e8 // per))))
    children = _log(rng, 1, 96)
    return dict(kind="cow", model=model, children=children, donors=rng.randint(1, children))


# ------------------------------------------------------------------ inputs

def _lengths(n, lo, hi, mix):
    return np.random.default_rng(mix).integers(lo, hi + 1, n).astype(np.int64)


class _State:
    """Buffers by name, the launches of a pass, and the graph that replays them."""


_STREAMS = {}


def _stream(nova):
    # one stream per library: passes follow each other, as a program's steps do
    if nova.model not in _STREAMS:
        _STREAMS[nova.model] = nova.dev_stream_create()
    return _STREAMS[nova.model]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, shape, scale=1.0, dtype=torch.float32):
    x = torch.empty(shape, dtype=dtype, device="cuda")
    x.normal_(0.0, scale, generator=g)
    return x


def _dev(array):
    return torch.from_numpy(np.ascontiguousarray(array)).cuda()


def _capture(s, nova, launches):
    """Record a pass's launches into a graph."""
    stream = _stream(nova)
    nova.dev_graph_begin(stream)
    launches(stream)
    graph = nova.dev_graph_end(stream)
    weakref.finalize(s, nova.dev_graph_destroy, graph)
    s.replay = lambda: nova.dev_graph_launch(graph, stream)


def _paged(s, seed, case, lengths):
    """Pools of `layers` layers, one block table per session over shuffled pages."""
    nkv = MODELS[case["model"]][1]
    pages = (lengths + KB - 1) // KB
    s.nb = int(pages.sum()) + 8
    perm = np.random.default_rng(seed).permutation(s.nb).astype(np.int32)
    s.stride = int(pages.max())
    table = np.zeros((len(pages), s.stride), np.int32)
    off = 0
    for i, p in enumerate(pages):
        table[i, :p] = perm[off:off + p]
        off += int(p)
    s.table_host, s.table = table, _dev(table)
    g = _gen(seed)
    shape = (case["layers"], s.nb, KB, nkv, HD)
    s.pool_k = _normal(g, shape, 1.0, torch.float16)
    s.pool_v = _normal(g, shape, 1.0, torch.float16)
    return g


def _rope_tables(nova, rows):
    cs = torch.empty((rows, HALF), device="cuda")
    sn = torch.empty((rows, HALF), device="cuda")
    nova.launch_rope_table_rows(cs.data_ptr(), sn.data_ptr(), rows, None)
    return cs, sn


def _inputs(case, seed):
    """The tensors of a case, before anything ran on them."""
    s = _State()
    s.case = case
    nh, nkv, _ = MODELS[case["model"]]
    if case["kind"] == "decode":
        n, layers = case["sessions"], case["layers"]
        s.ctx = _lengths(n, case["ctx_lo"], case["ctx_hi"], case["mix"])
        g = _paged(s, seed, case, s.ctx + 1)
        # post-RoPE queries are not unit scale: scores spread over several units
        s.q = _normal(g, (layers, n, nh, HD), 2.0)
        half = case["form"] == "planned"
        s.k_new = _normal(g, (layers, n, nkv, HD), 1.0, torch.float16 if half else torch.float32)
        s.v_new = _normal(g, (layers, n, nkv, HD), 1.0, torch.float16 if half else torch.float32)
    elif case["kind"] == "prefill":
        n, layers, n_q = case["sessions"], case["layers"], case["n_q"]
        s.ctx = _lengths(n, case["past_lo"], case["past_hi"], case["mix"])
        g = _paged(s, seed, case, s.ctx + n_q)
        s.q = _normal(g, (layers, n, n_q, nh, HD), 2.0)
        s.k_new = _normal(g, (layers, n, n_q, nkv, HD))
        s.v_new = _normal(g, (layers, n, n_q, nkv, HD))
    elif case["kind"] == "gemv":
        g = _gen(seed)
        s.w = []
        for _ in range(case["layers"]):
            s.w.append({name: _q4k(g, rows, cols) for name, (rows, cols) in _projections(case).items()})
        layers, t = case["layers"], case["tokens"]
        s.x = _normal(g, (layers, 3, t, case["hidden"]))         # inputs of q/k/v, of o and of gate/up
        s.act = _normal(g, (layers, t, case["ffn"]))             # input of down
    else:
        layers = MODELS[case["model"]][2]
        g = _gen(seed)
        order = np.random.default_rng(seed).permutation(case["donors"] + case["children"]).astype(np.int32)
        s.nb = len(order)
        s.src = order[np.arange(case["children"]) % case["donors"]]
        s.dst = order[case["donors"]:]
        s.pool_k = _normal(g, (layers, s.nb, KB, nkv, HD), 1.0, torch.float16)
        s.pool_v = _normal(g, (layers, s.nb, KB, nkv, HD), 1.0, torch.float16)
        s.table = torch.zeros(case["children"], dtype=torch.int32, device="cuda")
    return s


def _projections(case):
    """rows x cols of a layer's seven Q4_K matrices."""
    hidden, kv, ffn = case["hidden"], case["kv"], case["ffn"]
    return {"q": (hidden, hidden), "k": (kv, hidden), "v": (kv, hidden), "o": (hidden, hidden), "gate": (ffn, hidden),
            "up": (ffn, hidden), "down": (hidden, ffn)}


def _q4k(g, rows, cols):
    """Random ggml block_q4_K blocks: fp16 scale and min, 12 B of 6-bit scales, 128 B of nibbles."""
    b = torch.randint(0, 256, (rows, cols // 256, 144), dtype=torch.uint8, device="cuda", generator=g)
    d = torch.empty((rows, cols // 256, 2), device="cuda")
    d[..., 0].uniform_(2e-4, 4e-3, generator=g)
    d[..., 1].uniform_(1e-4, 2e-3, generator=g)
    b[..., 0:4] = d.to(torch.float16).view(torch.uint8)
    return b


# ------------------------------------------------------------------ passes

def prepare(case, seed):
    nova = nova_amd.load(case["model"])
    s = _inputs(case, seed)
    {"decode": _prepare_decode, "prefill": _prepare_prefill, "gemv": _prepare_gemv, "cow": _prepare_cow}[case["kind"]](
        nova, s, case)
    torch.cuda.synchronize()
    return s


def _prepare_decode(nova, s, case):
    n, form = case["sessions"], case["form"]
    s.n_keys = _dev((s.ctx + 1).astype(np.int32))
    s.o = torch.empty_like(s.q)
    pk, pv, tab, nk = s.pool_k.data_ptr(), s.pool_v.data_ptr(), s.table.data_ptr(), s.n_keys.data_ptr()
    if form != "planned":
        s.cs, s.sn = _rope_tables(nova, int(s.ctx.max()) + 1)
        cs, sn = s.cs.data_ptr(), s.sn.data_ptr()
    if form in ("planned", "rope"):
        s.ws = torch.empty(nova.attn_decode_batch_workspace_bytes(n), dtype=torch.uint8, device="cuda")
        ws = s.ws.data_ptr()
    if form == "calls":
        s.scratch = torch.empty(nova.nh * 32 * (HD + 2), device="cuda")

    def launches(st):
        if form in ("planned", "rope"):
            nova.launch_attn_decode_plan(tab, s.stride, nk, n, ws, st)
        for layer in range(case["layers"]):
            q, o = s.q[layer].data_ptr(), s.o[layer].data_ptr()
            k, v = s.k_new[layer].data_ptr(), s.v_new[layer].data_ptr()
            if form == "planned":
                nova.launch_attn_decode_paged_planned(q, pk, pv, tab, s.stride, n, layer, s.nb, k, v, o, ws, st)
            elif form == "rope":
                nova.launch_attn_decode_paged_rope_planned(q, k, v, cs, sn, pk, pv, tab, s.stride, n, layer, s.nb, o,
                                                           ws, st)
            elif form == "rope_solo":
                nova.launch_attn_decode_paged_rope_solo(q, k, v, cs, sn, pk, pv, tab, s.stride, nk, n, layer, s.nb, o,
                                                        st)
            else:
                for i in range(n):
                    row = s.table[i].data_ptr()
                    nova.launch_rope_kv_store_paged(s.q[layer, i].data_ptr(), s.k_new[layer, i].data_ptr(),
                                                    s.v_new[layer, i].data_ptr(), cs, sn, pk, pv, row, layer, s.nb, 1,
                                                    int(s.ctx[i]), st)
                    nova.launch_attn_decode_paged(s.q[layer, i].data_ptr(), pk, pv, row, layer, s.nb,
                                                  int(s.ctx[i]) + 1, s.o[layer, i].data_ptr(), s.scratch.data_ptr(), st)

    _capture(s, nova, launches)


def _prepare_prefill(nova, s, case):
    n, n_q = case["sessions"], case["n_q"]
    s.n_past = _dev(s.ctx.astype(np.int32))
    s.o = torch.empty_like(s.q)
    s.cs, s.sn = _rope_tables(nova, int(s.ctx.max()) + n_q)
    cs, sn, pk, pv = s.cs.data_ptr(), s.sn.data_ptr(), s.pool_k.data_ptr(), s.pool_v.data_ptr()

    def launches(st):
        for layer in range(case["layers"]):
            if case["form"] == "batch":
                nova.launch_rope_kv_store_paged_batch(s.q[layer].data_ptr(), s.k_new[layer].data_ptr(),
                                                      s.v_new[layer].data_ptr(), cs, sn, pk, pv, s.table.data_ptr(),
                                                      s.stride, s.n_past.data_ptr(), n, n_q, layer, s.nb, st)
                nova.launch_attn_prefill_paged_batch(s.q[layer].data_ptr(), pk, pv, s.table.data_ptr(), s.stride,
                                                     s.n_past.data_ptr(), n, n_q, layer, s.nb, s.o[layer].data_ptr(),
                                                     st)
                continue
            for i in range(n):
                row, past = s.table[i].data_ptr(), int(s.ctx[i])
                nova.launch_rope_kv_store_paged(s.q[layer, i].data_ptr(), s.k_new[layer, i].data_ptr(),
                                                s.v_new[layer, i].data_ptr(), cs, sn, pk, pv, row, layer, s.nb, n_q,
                                                past, st)
                nova.launch_attn_prefill_paged(s.q[layer, i].data_ptr(), pk, pv, row, layer, s.nb, n_q, past,
                                               s.o[layer, i].data_ptr(), st)

    _capture(s, nova, launches)


def _prepare_gemv(nova, s, case):
    shapes, t = _projections(case), case["tokens"]
    layers, hidden, ffn = case["layers"], case["hidden"], case["ffn"]
    s.out = {name: torch.empty((layers, t, rows), device="cuda") for name, (rows, _) in shapes.items()}

    def q8(n):
        # ActQ8 of one activation: codes, scales per 32, sums per 16
        return (torch.empty((layers, t, n), dtype=torch.int8, device="cuda"),
                torch.empty((layers, t, n // 32), device="cuda"),
                torch.empty((layers, t, n // 16), dtype=torch.int32, device="cuda"))

    s.q8 = {"down": q8(ffn)}
    if t == 4:
        s.q8.update(qkv=q8(hidden), o=q8(hidden), gate_up=q8(hidden))
    groups = (("qkv", ("q", "k", "v")), ("o", ("o",)), ("gate_up", ("gate", "up")))

    def launches(st):
        for layer in range(layers):
            def quant(act, x):
                qs, d, sums = (a[layer].data_ptr() for a in s.q8[act])
                nova.launch_quant_q8(qs, d, sums, x.data_ptr(), t, x.shape[-1], st)
                return qs, d, sums

            for i, (act, names) in enumerate(groups):
                if t == 1:
                    k = len(names)
                    nova.launch_gemv_q4k_f32(
                        (ctypes.c_void_p * k)(*[s.w[layer][m].data_ptr() for m in names]),
                        (ctypes.c_int64 * k)(*[shapes[m][0] for m in names]),
                        (ctypes.c_void_p * k)(*[s.out[m][layer].data_ptr() for m in names]),
                        k, hidden, s.x[layer, i].data_ptr(), st)
                    continue
                codes = quant(act, s.x[layer, i])
                for m in names:
                    nova.launch_gemv4_q4k(s.w[layer][m].data_ptr(), shapes[m][0], hidden, *codes,
                                          s.out[m][layer].data_ptr(), st)
            codes = quant("down", s.act[layer])
            gemv = nova.launch_gemv_q4k if t == 1 else nova.launch_gemv4_q4k
            gemv(s.w[layer]["down"].data_ptr(), shapes["down"][0], ffn, *codes, s.out["down"][layer].data_ptr(), st)

    _capture(s, nova, launches)


def _prepare_cow(nova, s, case):
    n = case["children"]
    ops = (nova_amd.CowOp * n)(*[nova_amd.CowOp(int(a), int(b), i) for i, (a, b) in enumerate(zip(s.src, s.dst))])
    stream = _stream(nova)
    pk, pv, tab = s.pool_k.data_ptr(), s.pool_v.data_ptr(), s.table.data_ptr()
    s.replay = lambda: nova.launch_kv_cow_apply(pk, pv, s.nb, tab, ops, n, stream)


def run(state):
    state.replay()
    kind = state.case["kind"]
    if kind == "decode":
        out = {"o": state.o, "pool_k": state.pool_k.view(torch.int16), "pool_v": state.pool_v.view(torch.int16)}
        if state.case["form"] == "calls":
            out["q"] = state.q
        return out
    if kind == "prefill":
        return {"o": state.o, "q": state.q, "pool_k": state.pool_k.view(torch.int16),
                "pool_v": state.pool_v.view(torch.int16)}
    if kind == "gemv":
        return {"out": state.out, "q8": state.q8}
    return {"pool_k": state.pool_k.view(torch.int16), "pool_v": state.pool_v.view(torch.int16), "table": state.table}


# ------------------------------------------------------------------ work and tolerance

def work(case):
    nh, nkv, n_layers = MODELS[case["model"]]
    if case["kind"] == "decode":
        keys = _lengths(case["sessions"], case["ctx_lo"], case["ctx_hi"], case["mix"]) + 1
        row = nkv * HD
        new = 2 if case["form"] == "planned" else 4
        per = int((keys - 1).sum()) * row * 4 + len(keys) * (row * 2 * new + row * 4 + nh * HD * 8)
        per += int(((keys + KB - 1) // KB).sum()) * 4
        return {"bytes": case["layers"] * per, "flops": case["layers"] * int(keys.sum()) * nh * HD * 4}
    if case["kind"] == "prefill":
        past, n_q = _lengths(case["sessions"], case["past_lo"], case["past_hi"], case["mix"]), case["n_q"]
        pairs = int((past * n_q).sum()) + len(past) * n_q * (n_q + 1) // 2
        rows = int((past + n_q).sum()) * nkv * HD * 4                  # K and V of the prefix read, of the chunk written
        per = rows + len(past) * n_q * (nh * HD * 12 + nkv * HD * 8)   # q read and rotated, o written; new k, v read
        return {"bytes": case["layers"] * per, "flops": case["layers"] * pairs * nh * HD * 4}
    if case["kind"] == "gemv":
        shapes, t, hidden, ffn = _projections(case), case["tokens"], case["hidden"], case["ffn"]
        weights = sum(r * c // 256 * 144 for r, c in shapes.values())
        q8 = (ffn + (3 * hidden if t == 4 else 0)) * 11 // 8            # codes, scales and sums written
        per = weights + t * (4 * (3 * hidden + ffn) + q8 + 4 * sum(r for r, _ in shapes.values()))
        return {"bytes": case["layers"] * per, "flops": case["layers"] * t * 2 * sum(r * c for r, c in shapes.values())}
    page = n_layers * 2 * KB * nkv * HD * 2
    return {"bytes": (min(case["donors"], case["children"]) + case["children"]) * page, "flops": 0}


def tolerance(case):
    # fp16 pages, codes and tables are whole values: the same bits
    if case["kind"] == "cow":
        return "exact"
    # fp16 softmax weights: measured 0.8e-4 to 1.8e-4 against 64 bits
    if case["kind"] == "prefill":
        return {"rel": 1e-3, "max": 0.03}
    # fp32-grade sums: measured below 1e-6 against 64 bits
    return {"rel": 1e-5, "max": 1e-3}


# ------------------------------------------------------------------ the results in 64 bits

def _rope_table64(rows):
    """The cos/sin table as it is defined: each step rounded to 32 bits."""
    i = torch.arange(HALF, dtype=torch.float32, device="cuda")
    l2 = torch.tensor(math.log2(THETA), dtype=torch.float64, device="cuda").to(torch.float32)
    f = torch.exp2((-i * (1.0 / HALF) * l2).double()).to(torch.float32)
    a = (torch.arange(rows, dtype=torch.float32, device="cuda")[:, None] * f).double()
    return torch.cos(a).to(torch.float32), torch.sin(a).to(torch.float32)


def _rotate(x, cs, sn):
    """NeoX pairs (i, i + 64) of the last dimension, in x's precision."""
    c, s = cs.to(x.dtype), sn.to(x.dtype)
    x0, x1 = x[..., :HALF], x[..., HALF:]
    return torch.cat([x0 * c - x1 * s, x0 * s + x1 * c], dim=-1)


def _attention64(q, k, v, first):
    """q [n_q][NH][HD] at positions first.. over keys k, v [n][NKV][HD] (fp16), in 64 bits."""
    n_q, nh, _ = q.shape
    n, nkv, _ = k.shape
    group = nh // nkv
    out = torch.empty((n_q, nh, HD), dtype=torch.float64, device="cuda")
    late = torch.arange(n, device="cuda")[None, :] > first + torch.arange(n_q, device="cuda")[:, None]
    late = late.repeat_interleave(group, 0)
    for h in range(nkv):
        qs = q[:, h * group:(h + 1) * group].double().reshape(n_q * group, HD)
        p = qs @ k[:, h].double().t().contiguous() / math.sqrt(HD)
        p = p.masked_fill_(late, -math.inf).softmax(-1)
        out[:, h * group:(h + 1) * group] = (p @ v[:, h].double().contiguous()).reshape(n_q, group, HD)
    return out


def exact(case, seed):
    s = _inputs(case, seed)
    if case["kind"] == "gemv":
        return _exact_gemv(s, case)
    if case["kind"] == "cow":
        return None
    chunk = case["kind"] == "prefill"
    n_q = case["n_q"] if chunk else 1
    rope = chunk or case["form"] != "planned"
    cs, sn = _rope_table64(int(s.ctx.max()) + n_q)
    q_out = torch.empty(s.q.shape, dtype=torch.float64, device="cuda")
    o = torch.empty_like(q_out)
    for layer in range(case["layers"]):
        pool_k = s.pool_k[layer].reshape(-1, *s.pool_k.shape[3:])
        pool_v = s.pool_v[layer].reshape(-1, *s.pool_v.shape[3:])
        for i in range(case["sessions"]):
            past = int(s.ctx[i])
            q, k, v = s.q[layer, i], s.k_new[layer, i], s.v_new[layer, i]
            if not chunk:
                q, k, v = q[None], k[None], v[None]
            q = q.double()
            if rope:
                c, sine = cs[past:past + n_q, None], sn[past:past + n_q, None]
                q, k = _rotate(q, c, sine), _rotate(k, c, sine)
            pos = np.arange(past)
            rows = _dev(s.table_host[i][pos // KB].astype(np.int64) * KB + pos % KB)
            # the new rows are stored as fp16 (nearest even) and attended as stored
            keys = torch.cat([pool_k[rows], k.to(torch.float16)])
            vals = torch.cat([pool_v[rows], v.to(torch.float16)])
            got = _attention64(q, keys, vals, past)
            o[layer, i] = got if chunk else got[0]
            q_out[layer, i] = q if chunk else q[0]
    out = {"o": o, "pool_k": None, "pool_v": None}
    if chunk or case["form"] == "calls":
        out["q"] = q_out
    return out


def _codes(x):
    """ActQ8 as it is defined, in 32 bits: codes and scales of 32 values each."""
    b = x.reshape(*x.shape[:-1], -1, 32)
    amax = b.abs().amax(-1, keepdim=True)
    # a division rounded once (a Python number over a tensor is a reciprocal and a product)
    inv = torch.where(amax > 0, torch.full_like(amax, 127.0) / amax, torch.zeros_like(amax))
    codes = torch.round(b * inv)
    return codes, (amax * torch.tensor(1.0 / 127.0, dtype=torch.float32, device="cuda")).squeeze(-1)


def _dequant64(b):
    """block_q4_K bytes [rows][n][144] as their weights in 64 bits."""
    d = b[..., 0:4].contiguous().view(torch.float16).double()
    sc = b[..., 4:16].to(torch.int32)
    low, high = sc[..., 0:4], sc[..., 4:8]
    scale = torch.cat([low & 63, (sc[..., 8:12] & 15) | ((low >> 6) << 4)], -1).double()
    least = torch.cat([high & 63, (sc[..., 8:12] >> 4) | ((high >> 6) << 4)], -1).double()
    nib = b[..., 16:].reshape(*b.shape[:-1], 4, 1, 32)
    q = torch.cat([nib & 15, nib >> 4], -2).reshape(*b.shape[:-1], 8, 32).double()
    w = d[..., 0:1, None] * scale[..., None] * q - d[..., 1:2, None] * least[..., None]
    return w.reshape(b.shape[0], -1)


def _exact_gemv(s, case):
    shapes = _projections(case)
    out = {name: torch.empty((case["layers"], case["tokens"], rows), dtype=torch.float64, device="cuda")
           for name, (rows, _) in shapes.items()}
    source = {"q": 0, "k": 0, "v": 0, "o": 1, "gate": 2, "up": 2}
    for layer in range(case["layers"]):
        for name, (rows, cols) in shapes.items():
            x = s.act[layer] if name == "down" else s.x[layer, source[name]]
            codes, scale = _codes(x)
            value = (codes.double() * scale.double()[..., None]).reshape(x.shape)
            for r in range(0, rows, 4096):
                w = _dequant64(s.w[layer][name][r:r + 4096])
                out[name][layer, :, r:r + 4096] = value @ w.t().contiguous()
    acts = ["down"] + (["qkv", "o", "gate_up"] if case["tokens"] == 4 else [])
    scales = {a: _codes(s.act if a == "down" else s.x[:, ("qkv", "o", "gate_up").index(a)])[1].double() for a in acts}
    return {"out": out, "q8": {a: (None, scales[a], None) for a in acts}}
