"""Workloads of the INT2 attention path, as a serving engine runs it, for timing and comparison.

A case is one engine step (metadata build and every layer's forward) through
``OscarMetadataBuilder`` and ``OscarAttentionImpl.forward``, or one call of the store:

* ``decode``: a uniform batch, one query token per request (or ``qlen`` of them: MTP
  verification). The layers are captured once in a HIP graph for a batch of ``slots`` requests,
  as vLLM does for the batches the builder declares graph support for; a step builds the
  metadata and replays it. Rows past the live requests are the graph's padding.
* ``chunk``: continuation chunks of a prompt over a cached prefix, with ``decodes`` one-token
  requests in the same step where chunked prefill mixes them. Plain launches.
* ``prefill``: first steps of requests without cached tokens. Plain launches.
* ``store``: K/V rotation, clip and INT2 packing of a batch of tokens.

The caches are written here in plain torch: records of rows that are Gaussian in the rotated
basis (what the calibrated rotations make of keys and values), clipped at the 96 % / 92 %
quantiles of the default configuration; queries are scaled so that scores spread by about two
nats, as trained attention does. Sizes: the configurations of ``bench.py`` (32 x 32768,
4 x 262144, the ragged MTP batch, 4 x 4096 prefill, 2048 tokens over 32768, the 4096-token
store) and generic ones around them. The calibration of the rotations runs once per model,
offline, and has no case.
"""

from __future__ import annotations

import math
from types import SimpleNamespace

import torch

DIM, PAGE, BLOCK, SLOT = 256, 768, 128, 160
DEV = "cuda"


# ------------------------------------------------------------------ the cases


def _step(name, kind, **over):
    case = dict(kind=kind, requests=1, slots=0, low=0, context=0, qlen=1, decodes=0, layers=1,
                group=6, kv_heads=1, sink=64, recent=256, spec=3, clip="percentile")
    case.update(over)
    return dict(case, name=name) if name else case


def listed():
    return [
        # One user, a short conversation: the smallest decode step, launches and latency.
        _step("decode 1x700", "decode", requests=1, slots=1, low=700, context=700, layers=4),
        # One user deep into a long document: little parallel work outside the split history.
        _step("decode 1x100k", "decode", requests=1, slots=1, low=100003, context=100003, layers=4),
        # A chat server's batch: ragged lengths, a graph of 128 slots with 117 requests live.
        _step("decode 117 ragged", "decode", requests=117, slots=128, low=300, context=12000,
              layers=4),
        # The headline decode: 32 requests of 32768 tokens on one tensor-parallel rank.
        _step("decode 32x32k", "decode", requests=32, slots=32, low=32768, context=32768,
              layers=4, sink=4, recent=128),
        # Long context: 4 requests of 262144 tokens.
        _step("decode 4x262k", "decode", requests=4, slots=4, low=262144, context=262144,
              layers=4, sink=4, recent=128),
        # MTP verification of a few users: 4 query tokens each over about 9k tokens.
        _step("mtp 7x9k", "decode", requests=7, slots=8, low=6001, context=12007, qlen=4, layers=4),
        # Ragged MTP batch: 64 requests, 256 to 131072 tokens, 4 query tokens each.
        _step("mtp 64 ragged", "decode", requests=64, slots=64, low=256, context=131072, qlen=4,
              layers=4, sink=4, recent=128),
        # A long prompt's next chunk: 2048 tokens over 32768 cached ones.
        _step("chunk 2048 over 32k", "chunk", context=32768, qlen=2048, sink=4, recent=128),
        # Chunked prefill beside decoding: 389 tokens of a prompt over 20011, 15 decodes.
        _step("chunk 389 + 15 decodes", "chunk", context=20011, qlen=389, decodes=15, low=1500,
              layers=2),
        # Prompts that arrive together: 4 requests of 4096 tokens.
        _step("prefill 4x4096", "prefill", requests=4, low=4096, context=4096, sink=4, recent=128),
        # Short prompts of odd lengths, two KV heads on the rank.
        _step("prefill 9 ragged", "prefill", requests=9, low=33, context=1201, layers=2, kv_heads=2,
              group=4),
        # The INT2 store of a prefill batch with the 8-factor clip search.
        _step("store 16k search", "store", qlen=16384, clip="search", sink=4, recent=128),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "mtp", "mtp", "chunk", "chunk", "prefill", "store"])
    short = rng.random() < 0.4
    over = dict(group=rng.choice([6, 6, 6, 4, 5, 8]), kv_heads=rng.choice([1, 1, 1, 2]),
                sink=4 if short else 64, recent=128 if short else 256)
    heads = over["kv_heads"]
    if kind in ("decode", "mtp"):
        qlen = 1 if kind == "decode" else rng.choice([2, 3, 4, 4])
        requests = _log(rng, 1, 128 if qlen == 1 else 64)
        most = min(262144, (1 << 20) // (requests * heads))
        context = _log(rng, 300, max(301, most))
        low = context if rng.random() < 0.4 else max(260, context // rng.choice([2, 8, 40]))
        slots = next(s for s in (1, 2, 4, 8, 16, 24, 32, 48, 64, 96, 128) if s >= requests)
        return _step("", "decode", requests=requests, slots=slots, low=min(low, context),
                     context=context, qlen=qlen, layers=4, **over)
    if kind == "chunk":
        qlen = _log(rng, 20, 2048)
        requests = 1 if qlen > 700 else rng.choice([1, 1, 2, 3])
        decodes = rng.choice([0, 0, 3, 20])
        rows = (qlen * requests + decodes) * over["group"] * heads
        layers = 2 if rows < 3000 else 1
        context = _log(rng, 400, min(131072, max(401, 11000 * 32768 // (rows * layers) - qlen)))
        return _step("", "chunk", requests=requests, context=context, qlen=qlen, decodes=decodes,
                     low=min(context, 500), layers=layers, **over)
    if kind == "prefill":
        requests = _log(rng, 1, 16)
        rows = over["group"] * heads * requests
        context = _log(rng, 30, min(8192, int(math.sqrt(24 * 4096 * 4096 / rows))))
        return _step("", "prefill", requests=requests, low=max(20, context // rng.choice([1, 3, 10])),
                     context=context, layers=2 if rows * context < 20000 else 1, **over)
    over.update(group=6, kv_heads=1)
    return _step("", "store", qlen=_log(rng, 64, 16384),
                 clip=rng.choice(["percentile", "factor", "search"]), **over)


def _requests(case):
    """(cached tokens, query tokens) of each request, the same for every seed: lengths spread
    over the logarithm from low to context."""
    n, low, high = case["requests"], case["low"], case["context"]
    spread = [int(round(low * (high / low) ** ((i + 0.5) / max(n, 1)))) if low else 0
              for i in range(n)]
    if case["kind"] == "decode":
        return [(max(0, s - case["qlen"]), case["qlen"]) for s in spread]
    if case["kind"] == "prefill":
        return [(0, s) for s in spread]
    d = case["decodes"]
    lengths = [int(round(low * (high / low) ** ((i + 0.5) / d))) for i in range(d)]
    return [(s - 1, 1) for s in lengths] + [(case["context"], case["qlen"])] * n


def _parts(case, prefix):
    """(sink tokens, first recent token) of a request with ``prefix`` cached tokens: INT2
    history lies between them, the window holds the others."""
    sink = min(case["sink"], prefix)
    return sink, max(sink, prefix - case["recent"])


def work(case):
    """What a pass cannot do without: 136 bytes per INT2 history token-head and 1024 per BF16
    window token-head read, q, k, v read, the output, the new records (136) and window rows
    written, the block table; 4 operations per query row, visible key and dim, and the
    rotations of q, k, v and the history output."""
    heads, rows = case["kv_heads"], case["kv_heads"] * case["group"]
    rotate = 2 * DIM * DIM
    if case["kind"] == "store":
        n = case["qlen"] * heads
        return {"bytes": n * (1024 + 136) + case["qlen"] * 8 + 4 * DIM * DIM,
                "flops": n * 2 * rotate}
    ring = case["recent"] + case["spec"] + 1
    total = flops = 0
    for prefix, n in _requests(case):
        sink, recent = _parts(case, prefix)
        hist, window = recent - sink, sink + prefix - recent
        total += heads * (136 * hist + 1024 * window + n * (1024 + 136)) + n * 8
        total += heads * 1024 * min(n, case["sink"] + ring) + 4 * -(-(prefix + n) // BLOCK)
        total += n * rows * DIM * 4
        flops += rows * DIM * 4 * (n * prefix + n * (n + 1) // 2)
        flops += n * rotate * (2 * heads + (2 * rows if prefix else 0))
    return {"bytes": case["layers"] * total, "flops": case["layers"] * flops}


# Four times the largest difference between the layer step and its 64-bit value, over the
# listed and drawn cases. Bytes (records, window rows) are equal.
def tolerance(case):
    if case["kind"] == "store":
        return "exact"
    if case["kind"] == "prefill":
        return {"rel": 0.01, "max": 0.2}
    return {"rel": 0.02, "max": 0.4}


# ------------------------------------------------------------------ inputs


def _rotation(gen):
    return torch.linalg.qr(torch.randn(DIM, DIM, generator=gen, device=DEV))[0].bfloat16()


def _records(n, gen):
    """[n, 160] uint8 records of Gaussian rows: 2-bit codes, fp16 scale and zero, of K, then V."""
    out = torch.zeros(n, SLOT, dtype=torch.uint8, device=DEV)
    for at, clip in ((0, 2.05), (68, 1.75)):
        x = torch.randn(n, DIM, generator=gen, device=DEV)
        x.clamp_(-clip, clip)
        low = x.amin(1, keepdim=True)
        scale = ((x.amax(1, keepdim=True) - low) / 3).half()
        low = low.half()
        x.sub_(low.float()).div_(scale.float()).round_().clamp_(0, 3)
        codes = x.to(torch.uint8).view(n, DIM // 4, 4)
        out[:, at : at + 64] = (codes[..., 0] | codes[..., 1] << 2 | codes[..., 2] << 4
                                | codes[..., 3] << 6)
        out[:, at + 64 : at + 68] = torch.cat([scale, low], 1).view(torch.uint8)
    return out


def _tables(requests, gen):
    """Pages of every request and the pool's size. Page 0 is nobody's, the first pages lie at
    the pool's start, the last ones (the newest) at its end, the others anywhere between."""
    need = [-(-(p + n) // PAGE) for p, n in requests]
    count = len(need)
    middle = sum(max(0, n - 2) for n in need)
    pool = 1 + 2 * count + middle + middle // 8
    shuffle = lambda n: torch.randperm(n, generator=gen, device=DEV).cpu()  # noqa: E731
    first, last = 1 + shuffle(count), pool - count + shuffle(count)
    others = 1 + count + shuffle(pool - 1 - 2 * count)
    pages, at = [], 0
    for r, n in enumerate(need):
        inner = others[at : at + max(0, n - 2)]
        at += max(0, n - 2)
        pages.append(torch.cat([first[r : r + 1], inner, last[r : r + 1] if n > 1 else last[:0]]))
    return pages, pool, count


def _inputs(case, seed):
    """A step's inputs in plain torch: caches, tables, rotations and rows of every layer."""
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    heads, group, layers = case["kv_heads"], case["group"], case["layers"]
    requests = _requests(case)
    pages, pool, count = _tables(requests, gen)
    ring = case["recent"] + case["spec"] + 1
    stripe = PAGE * heads * DIM * 2
    tokens = max(sum(n for _, n in requests), case["slots"] * case["qlen"])
    w = SimpleNamespace(case=case, requests=requests, pages=pages, pool=pool, count=count,
                        tokens=tokens, layers=[])
    for _ in range(layers):
        k_cache = torch.zeros(pool * PAGE // BLOCK, BLOCK, heads, DIM, dtype=torch.bfloat16,
                              device=DEV)
        v_cache = torch.zeros_like(k_cache)
        records = k_cache.view(torch.uint8).view(pool, stripe)
        window = v_cache.view(pool, -1)
        for (prefix, _), own in zip(requests, pages):
            if not prefix:
                continue
            own = own.to(DEV)[: -(-prefix // PAGE)]
            rows = _records(own.numel() * PAGE * heads, gen).view(own.numel(), -1)
            records[own, : PAGE * heads * SLOT] = rows
            live = case["sink"] + ring
            window[own[0], : live * 2 * heads * DIM] = torch.randn(
                live * 2 * heads * DIM, generator=gen, device=DEV).bfloat16()
        w.layers.append(SimpleNamespace(
            k_cache=k_cache, v_cache=v_cache, rk=_rotation(gen), rv=_rotation(gen),
            q=(2 * torch.randn(tokens, heads * group, DIM, generator=gen, device=DEV)).bfloat16(),
            k=torch.randn(tokens, heads, DIM, generator=gen, device=DEV).bfloat16(),
            v=torch.randn(tokens, heads, DIM, generator=gen, device=DEV).bfloat16(),
            out=torch.zeros(tokens, heads * group * DIM, dtype=torch.bfloat16, device=DEV)))
    return w


def _table(w):
    per = PAGE // BLOCK
    table = torch.zeros(max(len(w.pages), w.case["slots"]), max(len(p) for p in w.pages) * per,
                        dtype=torch.int32)
    for r, own in enumerate(w.pages):
        table[r, : len(own) * per] = (own[:, None] * per + torch.arange(per)).reshape(-1)
    return table


def _common(w, table, requests, slots):
    """The scheduler's metadata of one step, as vLLM hands it to the builder."""
    starts = torch.tensor([0] + [n for _, n in requests]).cumsum(0).to(torch.int32)
    lengths = torch.tensor([p + n for p, n in requests], dtype=torch.int32)
    return SimpleNamespace(
        query_start_loc=starts.to(DEV), query_start_loc_cpu=starts, seq_lens=lengths.to(DEV),
        seq_lens_cpu=lengths, num_reqs=len(requests), num_actual_tokens=int(starts[-1]),
        max_query_len=max(n for _, n in requests), max_seq_len=int(lengths.max()),
        block_table_tensor=table.to(DEV), slot_mapping=slots, causal=True,
        attn_state="PrefillNoCache" if w.case["kind"] == "prefill" else "ChunkedPrefill")


def _config(case):
    from oscar_new_amd.config import OscarConfig

    return OscarConfig(sink_tokens=case["sink"], recent_tokens=case["recent"],
                       speculative_tokens=case["spec"], clip_mode=case["clip"])


def _store_inputs(case, seed):
    """K/V rows with a few outlier channels and permuted 128-token pages."""
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    n, heads = case["qlen"], case["kv_heads"]
    scale = torch.ones(DIM, device=DEV)
    scale[torch.randperm(DIM, generator=gen, device=DEV)[:5]] = 10
    rows = [(torch.randn(n, heads, DIM, generator=gen, device=DEV) * scale).bfloat16()
            for _ in range(2)]
    pool = -(-n // PAGE) + 2
    blocks = torch.randperm(pool * PAGE // BLOCK, generator=gen, device=DEV)[: -(-n // BLOCK)]
    slots = (blocks[:, None] * BLOCK + torch.arange(BLOCK, device=DEV)).reshape(-1)[:n].contiguous()
    history = torch.zeros(pool * PAGE * heads * DIM * 2, dtype=torch.uint8, device=DEV)
    rt = [_rotation(gen).T.contiguous() for _ in range(2)]
    return rows, rt, history, slots, torch.tensor([1, n], dtype=torch.int32, device=DEV)


def prepare(case, seed):
    from oscar_new_amd.backend import OscarAttentionImpl
    from oscar_new_amd.layout import CacheLayout
    from oscar_new_amd.metadata import OscarMetadataBuilder

    layout = CacheLayout(PAGE, kv_heads=case["kv_heads"], config=_config(case))
    if case["kind"] == "store":
        rows, rt, history, slots, counts = _store_inputs(case, seed)
        return SimpleNamespace(case=case, layout=layout, rows=rows, rt=rt, history=history,
                               slots=slots, counts=counts)
    w = _inputs(case, seed)
    table = _table(w)
    slots = torch.cat([table[r][torch.arange(p, p + n) // BLOCK].long() * BLOCK
                       + torch.arange(p, p + n) % BLOCK for r, (p, n) in enumerate(w.requests)])
    w.common = _common(w, table, w.requests, slots.to(DEV))
    batch = max(len(w.requests), case["slots"])
    w.builder = OscarMetadataBuilder.standalone(layout, batch, w.tokens, table.shape[1] * BLOCK, DEV)
    for layer in w.layers:
        layer.impl = OscarAttentionImpl.standalone(case["kv_heads"] * case["group"], DIM, 1 / 16,
                                                   case["kv_heads"], layout.config)
        layer.impl.set_rotations(layer.rk, layer.rv)
    w.graph = None
    if case["kind"] == "decode":  # captured for the padded batch, before any request is there
        uniform = [(0, case["qlen"])] * case["slots"]
        dummy = _common(w, table, uniform, torch.full((w.tokens,), -1, device=DEV))
        meta = w.builder.build_for_cudagraph_capture(dummy)
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _forward(w, meta)
        torch.cuda.current_stream().wait_stream(stream)
        w.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(w.graph, stream=stream):
            _forward(w, meta)
    # What a step returns: outputs, and the pages that it writes to.
    end = w.pool - w.count
    w.outputs = []
    for layer in w.layers:
        records = layer.k_cache.view(torch.uint8).view(w.pool, -1)[:, : layout.history_page_bytes]
        window = layer.v_cache.view(w.pool, -1)[:, : layout.window_page_bytes // 2]
        w.outputs.append({"out": layer.out, "first": records[1 : 1 + w.count], "last": records[end:],
                          "window": window[1 : 1 + w.count]})
        if case["kind"] != "decode":  # long chunks write to any page
            w.outputs[-1]["records"] = records
    return w


def _forward(w, meta):
    for layer in w.layers:
        layer.impl.forward(None, layer.q, layer.k, layer.v, (layer.k_cache, layer.v_cache), meta,
                           layer.out)


def run(state):
    if state.case["kind"] == "store":
        from oscar_new_amd import kernels

        kernels.rotate_store_int2(*state.rows, *state.rt, state.history, state.slots, state.counts,
                                  state.layout)
        return state.history
    meta = state.builder.build(0, state.common)
    if state.graph is not None:
        state.graph.replay()
    else:
        _forward(state, meta)
    return state.outputs


# ------------------------------------------------------------------ 64-bit values


def _decoded(records):
    """(K, V) float64 rows of [n, 160] records."""
    rows = []
    for at in (0, 68):
        data = records[:, at : at + 64]
        codes = torch.stack([data >> s & 3 for s in (0, 2, 4, 6)], -1).reshape(-1, DIM).double()
        scale = records[:, at + 64 : at + 68].contiguous().view(torch.float16).double()
        rows.append(codes * scale[:, :1] + scale[:, 1:])
    return rows


def exact(case, seed):
    if case["kind"] == "store":
        return None
    w = _inputs(case, seed)
    heads, group, stripe = case["kv_heads"], case["group"], PAGE * case["kv_heads"] * DIM * 2
    ring = case["recent"] + case["spec"] + 1
    answers = []
    for layer in w.layers:
        records = layer.k_cache.view(torch.uint8).view(w.pool, stripe)
        window = layer.v_cache.view(w.pool, -1)
        rk, rv = layer.rk.double(), layer.rv.double()
        out = torch.zeros(w.tokens, heads * group, DIM, dtype=torch.float64, device=DEV)
        start = 0
        for (prefix, n), own in zip(w.requests, w.pages):
            sink, recent = _parts(case, prefix)
            own = own.to(DEV)
            at = torch.cat([torch.arange(sink), torch.arange(recent, prefix)]).to(DEV)
            at = torch.where(at < case["sink"], at, case["sink"] + at % ring)
            near = window[own[0], : (case["sink"] + ring) * 2 * heads * DIM].view(-1, 2, heads, DIM)
            near = near[at].double()
            far = records[own, : PAGE * heads * SLOT].reshape(-1, heads, SLOT)[sink:recent]
            tokens = slice(start, start + n)
            start += n
            for h in range(heads):
                old_k, old_v = _decoded(far[:, h])
                new_k = torch.cat([near[:, 0, h], layer.k[tokens, h].double()])
                new_v = torch.cat([near[:, 1, h], layer.v[tokens, h].double()])
                for g in range(h * group, (h + 1) * group):
                    for a in range(0, n, 1024):  # rows at a time: memory
                        b = min(n, a + 1024)
                        q = layer.q[tokens, g][a:b].double() / 16
                        seen = new_k.shape[0] - n + 1 + torch.arange(a, b, device=DEV)
                        score = q @ new_k.T
                        score.masked_fill_(torch.arange(new_k.shape[0], device=DEV)[None]
                                           >= seen[:, None], -math.inf)
                        p = torch.softmax(torch.cat([(q @ rk) @ old_k.T, score], 1), 1)
                        cut = recent - sink
                        out[tokens, g][a:b] = p[:, :cut] @ old_v @ rv.T + p[:, cut:] @ new_v
        answers.append({"out": out.view(w.tokens, -1), "first": None, "last": None, "window": None})
        if case["kind"] != "decode":
            answers[-1]["records"] = None
    return answers
