"""The BF16 branch of decode steps with few requests (blocks of 32 keys spread over the
workgroup's wavefronts, then merged) against the oracle's attention over the cache, at key
counts around a block, a round of four blocks and several rounds, with a wrapped ring, no
cached tokens and two KV heads; and the batch size from which the block-after-block form runs
(the same results within rounding)."""

import pytest
import torch

import oracle as O
from oscar_new_amd import kernels
from oscar_new_amd.backend import OscarAttentionImpl
from oscar_new_amd.config import OscarConfig
from tests._state import (assert_lse_close, assert_scaled_close, bits, make_state, native_views,
                          oracle_geometry, prepare_prefix)

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(lengths, out, lse, raw, layout, tables, prefixes, qs, ks, vs, rk, rv, pages=20):
    """Every request and KV head against the oracle's attention over the cache before the step."""
    k_cache, v_cache = native_views(raw, layout, pages)
    history = k_cache.reshape(-1).view(torch.uint8).cpu().numpy()
    window = bits(v_cache).reshape(-1)
    got = out.float().cpu().numpy().reshape(len(lengths), -1, 256)
    got_lse = lse.cpu().numpy()
    heads = layout.kv_heads
    g = got.shape[1] // heads
    for r, (n, p) in enumerate(zip(lengths, prefixes)):
        for h in range(heads):
            rows = slice(g * h, g * h + g)
            want, want_lse = O.cached_decode_reference(
                history, window, tables[r].numpy(), n, bits(qs[r][:, rows]), bits(ks[r][p:]),
                bits(vs[r][p:]), bits(rk), bits(rv), oracle_geometry(layout), 1 / 16, head=h)
            assert_scaled_close(got[r, rows], want, f"request {r} head {h}")
            assert_lse_close(got_lse[r, rows], want_lse[0], f"request {r} head {h} LSE")


def _step(lengths, cfg, kv_heads, seed, max_reqs, pages=20):
    g = torch.Generator().manual_seed(seed)
    prefixes = [n - 1 for n in lengths]
    hq = 4 * kv_heads
    layout, raw, hist, window, meta, tables = make_state(lengths, prefixes, cfg, pages=pages,
                                                         max_reqs=max_reqs, kv_heads=kv_heads)
    qr = lambda: torch.linalg.qr(torch.randn(256, 256, generator=g))[0].bfloat16().to(DEV)  # noqa: E731
    rk, rv = qr(), qr()
    ks = [torch.randn(n, kv_heads, 256, generator=g).bfloat16() for n in lengths]
    vs = [torch.randn(n, kv_heads, 256, generator=g).bfloat16() for n in lengths]
    # Scores of unit spread, for which the shared bounds are set: the oracle rounds dequantized
    # keys to bf16, which moves a score by its spread times 2^-9 / sqrt(3) and the output's
    # relative error with it (1.1 % measured at twice the spread, 0.5 % here).
    qs = [torch.randn(1, hq, 256, generator=g).bfloat16() for _ in lengths]
    prepare_prefix(ks, vs, rk, rv, hist, window, meta, tables, layout, prefixes)
    q = torch.cat(qs).to(DEV)
    k = torch.cat([x[p:] for x, p in zip(ks, prefixes)]).to(DEV)
    v = torch.cat([x[p:] for x, p in zip(vs, prefixes)]).to(DEV)
    meta.layout, meta.num_actual_tokens = layout, len(lengths)
    meta.merged_lse = torch.empty(len(lengths), hq, device=DEV)
    kernels.prepare_tasks(meta.query_start_loc, meta.counts, meta.tasks, meta.task_count,
                          meta.max_num_reqs, layout.config.queries_per_tile)
    impl = OscarAttentionImpl.standalone(hq, 256, 1 / 16, kv_heads, layout.config)
    impl.set_rotations(rk, rv)
    out = torch.empty(len(lengths), hq * 256, dtype=torch.bfloat16, device=DEV)
    before = raw.clone()
    impl.forward(None, q, k, v, native_views(raw, layout, pages), meta, out)
    torch.cuda.synchronize()
    return out, meta.merged_lse, before, layout, tables, prefixes, qs, ks, vs, rk, rv


@pytest.mark.parametrize("lengths,sink,recent,kv_heads", [
    ([1, 2, 31, 32, 33], 64, 256, 1),  # up to a block
    ([127, 128, 129, 161], 64, 256, 1),  # a round of four blocks, one block more
    ([320, 321, 322, 900], 64, 256, 2),  # the whole window, ring wrapped
    ([700, 1500], 4, 128, 2),
    ([700], 0, 0, 1),  # the current token alone
])
def test_decode_step_against_the_oracle(lengths, sink, recent, kv_heads):
    print(f"[raw waves] {lengths} S{sink} R{recent} H{kv_heads}", flush=True)
    cfg = OscarConfig(sink_tokens=sink, recent_tokens=recent)
    out, lse, raw, layout, tables, prefixes, qs, ks, vs, rk, rv = _step(lengths, cfg, kv_heads, 3, 8)
    _check(lengths, out, lse, raw, layout, tables, prefixes, qs, ks, vs, rk, rv)


@pytest.mark.parametrize("requests", [64, 65])
def test_both_sides_of_the_batch_rule(requests):
    # One (task, kv head) workgroup per request: 64 take the wavefront form, 65 the other.
    lengths = [200 + 3 * r for r in range(requests)]
    print(f"[raw waves] {requests} requests", flush=True)
    out, lse, raw, layout, tables, prefixes, qs, ks, vs, rk, rv = _step(
        lengths, OscarConfig(), 1, 4, requests, pages=80)
    _check(lengths, out, lse, raw, layout, tables, prefixes, qs, ks, vs, rk, rv, pages=80)
