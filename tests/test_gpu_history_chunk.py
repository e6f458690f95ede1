"""The history branch of continuation chunks (more than 16 query tokens per request: 128-row
tiles sharing each chunk's operands) against the dequantized cache in float64, split by split:
lengths around a tile's 128 rows and a chunk's 128 tokens, one and two KV heads, 4 to 8 query
heads per KV head, several splits (some empty), requests of one token beside a chunk (also in
batches whose task rows reach the token count, and with query tiles of 1 and 2), a request cut
short by the token count, and a history of more chunks than one table. The output buffers hold NaN
before the launch, so that a row that is not written fails.

Bounds: the shared attention bounds (relative L2 1e-2, LSE 1e-2) for scores of unit spread."""

import numpy as np
import pytest
import torch

from oscar_new_amd import kernels
from oscar_new_amd.backend import OscarAttentionImpl
from oscar_new_amd.config import OscarConfig
from tests._state import (assert_lse_close, assert_scaled_close, make_state, native_views,
                          prepare_prefix)

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _decoded(history, offsets):
    """(K, V) float64 rows of the 160-byte records at `offsets`."""
    rows = history[offsets[:, None] + torch.arange(160, device=DEV)]
    out = []
    for at in (0, 68):
        data = rows[:, at : at + 64]
        codes = torch.stack([data >> s & 3 for s in (0, 2, 4, 6)], -1).reshape(-1, 256).double()
        sz = rows[:, at + 64 : at + 68].contiguous().view(torch.float16).double()
        out.append(codes * sz[:, :1] + sz[:, 1:])
    return out


def _check(lengths, prefixes, splits, hq, kv_heads=1, sink=4, recent=128, pages=24, live=None,
           query_tile=4, max_reqs=8):
    cfg = OscarConfig(sink_tokens=sink, recent_tokens=recent, queries_per_tile=query_tile)
    torch.manual_seed(31)
    layout, raw, hist, window, meta, tables = make_state(lengths, prefixes, cfg, pages=pages,
                                                         kv_heads=kv_heads, max_reqs=max_reqs)
    eye = torch.eye(256, dtype=torch.bfloat16, device=DEV)
    ks = [torch.randn(n, kv_heads, 256).bfloat16() for n in lengths]
    vs = [torch.randn(n, kv_heads, 256).bfloat16() for n in lengths]
    prepare_prefix(ks, vs, eye, eye, hist, window, meta, tables, layout, prefixes)
    n = sum(a - b for a, b in zip(lengths, prefixes))
    q = torch.randn(n, hq, 256).bfloat16().to(DEV)
    kernels.prepare_tasks(meta.query_start_loc, meta.counts, meta.tasks, meta.task_count,
                          meta.max_num_reqs, cfg.queries_per_tile)
    if live is not None:
        meta.counts[1] = live
    with pytest.MonkeyPatch.context() as patch:
        patch.setattr(torch, "empty", lambda *a, **k: torch.full(*a, float("nan"), **k))
        got, lse = kernels.attention_partials(q, None, None, hist, window, meta, layout, 1 / 16,
                                              splits, raw=False, chunk=True)
    torch.cuda.synchronize()
    g, start = hq // kv_heads, 0
    for r, (length, prefix) in enumerate(zip(lengths, prefixes)):
        rows = slice(start, min(start + length - prefix, n if live is None else live))
        start += length - prefix
        prefix = length - (rows.stop - rows.start)  # as the kernels count a cut request's tokens
        s = min(sink, prefix)
        end = max(s, prefix - recent)
        per = -(-(-(-(end - s) // cfg.block_n)) // splits) * cfg.block_n
        slots = torch.tensor([int(tables[r, p // 128]) * 128 + p % 128 for p in range(s, end)],
                             dtype=torch.int64, device=DEV)
        for h in range(kv_heads):
            page, within = slots // layout.physical_block_tokens, slots % layout.physical_block_tokens
            k, v = _decoded(hist, page * layout.stripe_page_bytes + (within * kv_heads + h) * 160)
            x = q[rows, h * g : h * g + g].double() / 16
            for i in range(splits):
                part = got[rows, h * g : h * g + g, i].cpu().numpy()
                logs = lse[rows, h * g : h * g + g, i].cpu().numpy()
                a, b = min(i * per, end - s), min((i + 1) * per, end - s)
                if a == b:
                    assert not part.any() and np.isneginf(logs).all()
                    continue
                score = x @ k[a:b].T
                assert_scaled_close(part, (torch.softmax(score, -1) @ v[a:b]).cpu().numpy(),
                                    f"request {r} head {h} split {i}")
                assert_lse_close(logs, torch.logsumexp(score, -1).cpu().numpy(),
                                 f"request {r} head {h} split {i} LSE")


@pytest.mark.parametrize("lengths,prefixes,splits,hq,kv_heads", [
    ([217], [200], 1, 6, 1),  # 17 query tokens, 68 history tokens: less than a tile or chunk
    ([1044, 1043], [1023, 1022], 1, 6, 1),  # 126 rows: one tile
    ([1300], [1278], 3, 6, 1),  # 132 rows: 4 rows in the second tile
    ([388], [260], 2, 4, 1),  # exactly 128 history tokens, 512 rows
    ([2000], [389], 4, 5, 1),  # tiles that split a query's five heads
    ([1100, 700], [1000, 640], 2, 16, 2),  # two KV heads of eight
    ([900, 2500, 40, 1700], [899, 2499, 0, 1500], 5, 6, 1),  # decodes, a first chunk, a chunk
    ([3000], [2900], 16, 6, 1),
    ([300], [150], 8, 6, 1),  # 18 history tokens: empty splits
])
def test_partials_against_the_dequantized_cache(lengths, prefixes, splits, hq, kv_heads):
    print(f"[history chunk] {lengths} {prefixes} splits {splits} {hq}:{kv_heads}", flush=True)
    _check(lengths, prefixes, splits, hq, kv_heads)


@pytest.mark.parametrize("decodes,group,query_tile,max_reqs", [
    (133, 4, 4, 257),  # 134 tiles; as many task rows as tokens
    (250, 6, 4, 257),
    (256, 5, 4, 257),  # every request slot in use
    (26, 8, 2, 257),
    (3, 16, 1, 257),
    (5, 9, 1, 8),
])
def test_a_short_chunk_beside_many_decodes(decodes, group, query_tile, max_reqs):
    print(f"[history chunk] {decodes} decodes group {group} tile {query_tile}", flush=True)
    lengths = [210 + 7 * (i % 11) for i in range(decodes)] + [260]
    prefixes = [n - 1 for n in lengths[:-1]] + [243]
    _check(lengths, prefixes, 1, group, pages=decodes + 3, query_tile=query_tile,
           max_reqs=max_reqs)


def test_a_request_cut_short_by_the_token_count():
    print("[history chunk] cut short", flush=True)
    _check([900, 1300], [850, 1100], 2, 6, live=171)


@pytest.mark.parametrize("prefix", [131200, 131201, 280080])
def test_more_chunks_than_the_table_holds(prefix):
    # The record offsets of 1024 chunks of 128 tokens lie in LDS; the history starts in the first
    # chunk and ends 128 tokens before the prefix: the last chunk that fits, the next, 2188 chunks.
    print(f"[history chunk] {prefix} tokens", flush=True)
    _check([prefix + 20], [prefix], 1, 6, pages=(prefix + 20) // 768 + 3)


@pytest.mark.parametrize("lengths,prefixes,hq,kv_heads", [
    ([6100], [6000], 6, 1),  # a lone chunk, below and from 64 query tokens
    ([6030], [6000], 6, 1),
    ([9040, 700, 1500], [9000, 699, 1499], 8, 1),  # decodes beside it
    ([7050, 1300], [7000, 1299], 8, 2),
])
def test_steps_that_take_the_tile_kernel(lengths, prefixes, hq, kv_heads):
    """Layer steps whose host-side lengths select the kernel and several splits: the fused and the
    single launches carry the same bits, the task-shaped kernel's step agrees within rounding."""
    print(f"[history chunk] step {lengths} {hq}:{kv_heads}", flush=True)
    cfg = OscarConfig(sink_tokens=4, recent_tokens=128)
    torch.manual_seed(41)
    layout, raw, hist, window, meta, tables = make_state(lengths, prefixes, cfg, pages=24,
                                                         kv_heads=kv_heads)
    rot = [torch.linalg.qr(torch.randn(256, 256))[0].bfloat16().to(DEV) for _ in range(2)]
    ks = [torch.randn(n, kv_heads, 256).bfloat16() for n in lengths]
    vs = [torch.randn(n, kv_heads, 256).bfloat16() for n in lengths]
    prepare_prefix(ks, vs, *rot, hist, window, meta, tables, layout, prefixes)
    k, v = (torch.cat([x[p:] for x, p in zip(xs, prefixes)]).to(DEV) for xs in (ks, vs))
    n = k.shape[0]
    q = torch.randn(n, hq, 256).bfloat16().to(DEV)
    meta.layout, meta.num_actual_tokens = layout, n
    meta.max_seq_len, meta.total_seq_len = max(lengths), sum(lengths)
    meta.total_query_keys = sum((a - b) * a for a, b in zip(lengths, prefixes))
    kernels.prepare_tasks(meta.query_start_loc, meta.counts, meta.tasks, meta.task_count,
                          meta.max_num_reqs, cfg.queries_per_tile)

    def step(fused):
        impl = OscarAttentionImpl.standalone(hq, 256, 1 / 16, kv_heads, cfg, fused=fused)
        impl.set_rotations(*rot)
        splits, rule = impl.partition_for(meta)
        name = kernels.history_kernel_name(meta, layout, hq, n, rule, splits=splits)
        cache = raw.clone()
        meta.merged_lse = torch.full((n, hq), 7.0, device=DEV)
        out = torch.full((n, hq * 256), 3.0, device=DEV, dtype=torch.bfloat16)
        impl.forward(None, q, k, v, native_views(cache, layout, 24), meta, out)
        torch.cuda.synchronize()
        return (out.cpu(), meta.merged_lse.cpu(), cache.cpu()), name, splits

    got, name, splits = step(True)
    assert name == "history_chunk_kernel" and splits > 1
    for a, b in zip(got, step(False)[0]):
        assert torch.equal(a, b)
    meta.max_seq_len = None  # no host-side length
    want, name, splits = step(True)
    assert name != "history_chunk_kernel" and splits == 1
    assert torch.equal(got[2], want[2])
    for r in range(n):
        assert_scaled_close(got[0][r].float().numpy(), want[0][r].float().numpy(), f"row {r}")
    assert_lse_close(got[1].numpy(), want[1].numpy(), "merged LSE")
