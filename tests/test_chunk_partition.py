"""Host side of the continuation-chunk history launch, on the CPU: the split counts, the grid,
and the inline-asm copies of its kernel against the wait-state rule of the other kernels."""

import random
import subprocess
from pathlib import Path

import pytest

from oscar_new_amd import _ext
from oscar_new_amd.backend import OscarAttentionImpl
from oscar_new_amd.config import OscarConfig, attention_programs, choose_chunk_splits
from tests.test_isa_hazards import HIPCC, ROOT, _late_sites


@pytest.mark.parametrize("tokens,requests,heads,q_heads,longest,want", [
    (2048, 1, 1, 6, 34816, 5),  # 97 tiles: 485 of two rounds of 256 workgroups
    (389, 1, 1, 6, 20400, 13),
    (20, 1, 1, 6, 131072, 16),  # a tile or two: every split the one-round merge takes
    (17, 1, 1, 6, 100, 1),  # a single pipeline step
    (8192, 4, 2, 12, 2048, 1),  # tiles enough
    (2048, 1, 1, 6, None, 1),  # no host-side length
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
