"""The one-launch metadata fill against the copies and the task kernel it takes the place of:
the same buffers, byte for byte, and nothing written outside the step's part of them."""

from types import SimpleNamespace

import pytest
import torch

from oscar_new_amd import kernels
from oscar_new_amd.config import OscarConfig
from oscar_new_amd.layout import CacheLayout
from oscar_new_amd.metadata import OscarMetadataBuilder

pytestmark = pytest.mark.gpu
DEV = "cuda"
BUFFERS = ("qstarts", "seqs", "slots", "table", "counts", "tasks", "task_count")


def _builder():
    layout = CacheLayout(768, 1, config=OscarConfig(speculative_tokens=3))
    b = OscarMetadataBuilder.standalone(layout, 300, 4096, 40000, DEV)
    for name in BUFFERS:
        getattr(b, name).fill_(-7)
    return b


def _common(qlens, columns, max_seq_len, table_pad):
    g = torch.Generator().manual_seed(sum(qlens) + columns)
    nr, nt = len(qlens), sum(qlens)
    starts = torch.tensor([0] + list(qlens)).cumsum(0).to(torch.int32)
    table = torch.randint(0, 9999, (nr, columns + table_pad), generator=g, dtype=torch.int32)
    return SimpleNamespace(
        num_reqs=nr, num_actual_tokens=nt, max_query_len=max(qlens),
        query_start_loc=starts.to(DEV),
        seq_lens=torch.randint(1, 39000, (nr,), generator=g, dtype=torch.int32).to(DEV),
        block_table_tensor=table.to(DEV)[:, :columns],
        slot_mapping=torch.randint(-1, 1 << 40, (nt + 5,), generator=g).to(DEV),
        max_seq_len=max_seq_len, causal=True, attn_state=None)


# One request and one token; slot counts beside a workgroup's 1024; more requests than slot
# workgroups and the reverse; more requests than the 256 threads of a workgroup; padded table
# rows; a bounded and an unbounded column copy; a request without tokens.
@pytest.mark.parametrize("qlens,columns,max_seq_len,pad", [
    ([1], 1, 1, 0),
    ([1, 4, 3], 300, 39000, 0),
    ([1023], 17, None, 3),
    ([1024], 300, 129, 0),
    ([1000, 0, 25], 300, 128, 8),
    ([1] * 257, 257, 38000, 1),
    ([4] * 300, 313, None, 0),
    ([4001, 17, 5], 64, 8000, 0),
])
def test_one_launch_fill_equals_copies_and_task_kernel(qlens, columns, max_seq_len, pad):
    cm = _common(qlens, columns, max_seq_len, pad)
    a, b = _builder(), _builder()
    sources = (cm.query_start_loc, cm.seq_lens, cm.slot_mapping, cm.block_table_tensor)
    assert kernels.step_sources_fit(*sources, len(qlens), sum(qlens), a.counts.device)
    a.build(0, cm)
    # int64 query starts are converted by a tensor copy: the general path.
    cm.query_start_loc = cm.query_start_loc.to(torch.int64)
    assert not kernels.step_sources_fit(cm.query_start_loc, *sources[1:], len(qlens), sum(qlens),
                                        a.counts.device)
    b.build(0, cm)
    torch.cuda.synchronize()
    for name in BUFFERS:
        assert torch.equal(getattr(a, name), getattr(b, name)), name


def test_other_forms_take_the_general_path():
    cm = _common([1, 4, 3], 30, 3000, 0)
    sources = [cm.query_start_loc, cm.seq_lens, cm.slot_mapping, cm.block_table_tensor]
    dev = cm.seq_lens.device
    forms = {
        0: [sources[0][:3], sources[0].repeat_interleave(2)[::2], sources[0].cpu()],
        1: [sources[1].to(torch.int64), sources[1][:1].expand(3), sources[1].view(1, 3)],
        2: [sources[2].to(torch.int32), sources[2][:7], sources[2].repeat_interleave(2)[::2]],
        3: [sources[3][:2], sources[3].t().contiguous().t(), sources[3][:1].expand(3, 30)],
    }
    assert kernels.step_sources_fit(*sources, 3, 8, dev)
    for i, others in forms.items():
        for other in others:
            assert not kernels.step_sources_fit(*sources[:i], other, *sources[i + 1:], 3, 8, dev)


@pytest.mark.parametrize("requests,columns", [(0, 0), (0, 5), (2, 0)])
def test_steps_without_requests_or_columns(requests, columns):
    # Nothing to copy: empty tensors, which have no address.
    b = _builder()
    i32 = dict(dtype=torch.int32, device=DEV)
    starts = torch.arange(requests + 1, **i32)
    b.build(0, SimpleNamespace(
        num_reqs=requests, num_actual_tokens=requests, max_query_len=1, query_start_loc=starts,
        seq_lens=torch.ones(requests, **i32),
        block_table_tensor=torch.zeros((requests, columns), **i32),
        slot_mapping=torch.arange(requests, dtype=torch.int64, device=DEV), max_seq_len=None,
        causal=True, attn_state=None))
    assert b.counts.tolist() == [requests, requests] and b.task_count.item() == requests
