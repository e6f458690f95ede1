"""Host side of the continuation-chunk history launch, on the CPU: the split counts, the grid,
and the inline-asm copies of its kernel against the wait-state rule of the other kernels."""

import random
import subprocess
from pathlib import Path

import pytest

from oscar_new_amd import _ext, kernels
from oscar_new_amd.backend import OscarAttentionImpl
from oscar_new_amd.config import (OscarConfig, attention_programs, choose_chunk_splits,
                                  chunk_kernel_pays)
from oscar_new_amd.layout import CacheLayout
from tests.test_isa_hazards import HIPCC, ROOT, _late_sites


@pytest.mark.parametrize("tokens,requests,heads,q_heads,longest,want", [
    (2048, 1, 1, 6, 34816, 5),  # 97 tiles: 485 of two rounds of 256 workgroups
    (389, 1, 1, 6, 20400, 13),
    (20, 1, 1, 6, 131072, 16),  # a tile or two: every split the one-round merge takes
    (17, 1, 1, 6, 100, 1),  # a single pipeline step
    (8192, 4, 2, 12, 2048, 1),  # tiles enough
    (2048, 1, 1, 6, None, 1),  # no host-side length
    (8192, 1, 2, 12, 131072, 1),  # 128 MiB of split rows: a second split would pass it
    (8192, 1, 1, 6, 24192, 1),  # a third split would pass it
    (16384, 1, 1, 6, 262144, 1),
    (16384, 1, 4, 32, 262144, 1),  # one split alone passes it
])
def test_chunk_splits(tokens, requests, heads, q_heads, longest, want):
    assert choose_chunk_splits(tokens, requests, heads, q_heads, longest) == want


def test_long_chunks_take_the_chunk_splits():
    from types import SimpleNamespace

    meta = SimpleNamespace(num_reqs=1, num_actual_tokens=2048, max_query_len=2048, max_num_reqs=2,
                           max_seq_len=34816, layout=None)
    for policy, heads, want in (("device", 6, (5, 0)), ("mi355x", 6, (5, 0)),
                                ("reference", 6, (1, 0)), ("device", 2, (1, 0))):
        impl = OscarAttentionImpl.standalone(heads, 256, 1 / 16, 1, OscarConfig(),
                                             split_policy=policy)
        assert impl.partition_for(meta) == want


# Steps that were measured with both kernels, on both sides of the rule (layer step in us with the
# splits of choose_chunk_splits, and with the task-shaped kernel and one split).
@pytest.mark.parametrize("tokens,requests,group,heads,longest,total,pairs,tiles", [
    (2048, 1, 6, 1, 34816, None, None, True),  # 625, 810
    (94, 31, 6, 1, 16064, 218000, 1230000, True),  # 30 decodes: 150, 258
    (94, 31, 6, 1, 16064, 218000, None, True),
    (314, 251, 6, 1, 16064, 1700000, 2710000, False),  # 250 decodes: 370, 302
    (314, 251, 6, 1, 16064, None, None, False),
    (267, 251, 6, 1, 4017, 425000, 490000, False),  # 154, 109
    (124, 61, 4, 2, 16064, 420000, 1430000, False),  # 313, 183
    (300, 1, 6, 1, 800, 800, None, False),  # 112, 101
    (8192, 1, 6, 1, 24192, None, None, True),  # 1383, 1789
    (2078, 31, 6, 1, 10048, 111000, 20679000, True),  # 341, 436
    (404, 16, 6, 1, 20400, 117000, 8020000, True),
])
def test_steps_take_the_kernel_that_measured_faster(tokens, requests, group, heads, longest, total,
                                                    pairs, tiles):
    from types import SimpleNamespace

    cfg = OscarConfig()
    layout = CacheLayout(768, kv_heads=heads, config=cfg)
    meta = SimpleNamespace(num_reqs=requests, num_actual_tokens=tokens, max_query_len=64,
                           max_num_reqs=257, max_seq_len=longest, total_seq_len=total,
                           total_query_keys=pairs, layout=layout)
    impl = OscarAttentionImpl.standalone(group * heads, 256, 1 / 16, heads, cfg)
    splits, split_tokens = impl.partition_for(meta)
    name = kernels.history_kernel_name(meta, layout, group * heads, tokens, split_tokens,
                                       splits=splits)
    assert split_tokens == 0 and (name == "history_chunk_kernel") == tiles
    assert tiles or splits == 1
    # One split of a lone chunk leaves most CUs without a tile: the task-shaped kernel.
    assert kernels.history_kernel_name(meta, layout, group * heads, tokens) == (
        "history_chunk_kernel" if tokens == 8192 else
        "history_kernel<1>" if group == 4 else "history_w8_kernel")


def test_builder_sums_the_query_keys_of_chunk_steps(monkeypatch):
    from types import SimpleNamespace

    import torch

    from oscar_new_amd.metadata import OscarMetadataBuilder

    builder = OscarMetadataBuilder.standalone(CacheLayout(768, config=OscarConfig()), 4, 64, 4096,
                                              "cpu")
    monkeypatch.setattr(kernels, "prepare_tasks", lambda *a, **k: None)
    for lengths, tokens, want in (([900, 40000, 30], [1, 20, 3], 900 + 800000 + 90),
                                  ([900, 40000], [1, 4], None), ([500], [20], None)):
        starts = torch.tensor([0] + tokens).cumsum(0).to(torch.int32)
        lens = torch.tensor(lengths, dtype=torch.int32)
        meta = builder.build(0, SimpleNamespace(
            num_reqs=len(tokens), num_actual_tokens=sum(tokens), max_query_len=max(tokens),
            query_start_loc=starts, query_start_loc_cpu=starts, seq_lens=lens, seq_lens_cpu=lens,
            block_table_tensor=torch.zeros(len(tokens), 8, dtype=torch.int32),
            slot_mapping=torch.zeros(sum(tokens), dtype=torch.int64)))
        assert meta.total_query_keys == want


def test_no_host_side_length_keeps_the_task_shaped_kernel():
    assert not chunk_kernel_pays(2048, 1, 1, 6, 1, None)
    assert chunk_kernel_pays(2048, 1, 1, 6, 5, 34816)


def _tiles(lengths, query_tile, group):
    """128-row tiles that start in a task row of the requests, as the kernel finds them."""
    found = 0
    for tokens in lengths:
        for row0 in range(0, -(-tokens // query_tile) * query_tile * group, query_tile * group):
            b = -(-row0 // 128)
            found += b * 128 < row0 + query_tile * group
    return found


def _batches():
    """Chunks beside one-token decodes, up to the capacity, and ragged lengths."""
    rng = random.Random(17)
    for capacity in (1, 2, 17, 129, 257, 513, 1025):
        for decodes in {0, 1, 2, 26, 43, 116, 133, 160, 244, 256, 437, 512, 917, 1024}:
            if decodes < capacity:
                yield [1] * decodes + [17], capacity
                yield [1] * decodes + [64], capacity
        for _ in range(12):
            count = rng.randint(1, capacity)
            yield [rng.choice([0, 1, 1, 1, 2, 4, 5, 16, 17, 31, 33, 300]) for _ in range(count)] + [
                rng.choice([1, 17, 700])][: capacity - count], capacity


@pytest.mark.parametrize("query_tile,group", [(4, 4), (4, 5), (4, 6), (4, 8), (4, 1), (2, 6),
                                              (2, 8), (2, 16), (1, 9), (1, 12), (1, 16), (1, 32)])
def test_the_grid_holds_every_tile(query_tile, group):
    lib = _ext.library()
    for lengths, capacity in _batches():
        n = sum(lengths)
        if not n:
            continue
        programs = attention_programs(n, capacity, query_tile)
        grid = lib.oscar_history_chunk_tiles(n, capacity, programs, query_tile, group)
        need = _tiles(lengths, query_tile, group)
        assert need <= grid <= programs, (lengths, capacity)
        # A grid of exactly the task rows in use, too.
        tasks = sum(-(-t // query_tile) for t in lengths)
        grid = lib.oscar_history_chunk_tiles(n, capacity, tasks, query_tile, group)
        assert need <= grid <= tasks, (lengths, capacity)


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc is not installed")
def test_copies_keep_five_wait_states(tmp_path):
    out = tmp_path / "history_chunk.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17",
                    "-fno-gpu-flush-denormals-to-zero", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", f"-I{ROOT / 'include'}", "--cuda-device-only", "-S",
                    str(ROOT / "oscar_new_amd" / "csrc" / "history_chunk.hip"), "-o", str(out)],
                   check=True, capture_output=True, timeout=600)
    text = out.read_text()
    assert text.count("global_load_lds_dword") >= 6
    assert _late_sites(text) == []
