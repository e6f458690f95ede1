"""Rows of the BF16 branch whose scores are -inf (a key with an infinite element): p of such a
score is 0, also while a row has not met a finite score yet; a row that meets none is zero with
LSE -inf. Causal attention in float64 over the same bf16 inputs; the tolerances of the other
prefill comparisons (bf16 p and outputs: relative L2 1e-2, LSE 2e-2)."""

from types import SimpleNamespace

import pytest
import torch

from oscar_new_amd import kernels
from oscar_new_amd.config import OscarConfig
from oscar_new_amd.layout import CacheLayout

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n,infinite", [
    (1, [0]),  # one row, no finite score
    (40, list(range(35))),  # a whole block and rows of the next without a finite score
    (100, [0, 31, 32, 64, 99]),  # single keys at block edges, masked and unmasked blocks
    (700, list(range(0, 64)) + [300]),  # two blocks without a finite score, then finite ones
])
def test_minus_infinite_scores(n, infinite):
    print(f"[infinite scores] n {n}", flush=True)
    gen = torch.Generator().manual_seed(61)
    q = torch.randn(n, 6, 256, generator=gen).bfloat16()
    k = torch.randn(n, 1, 256, generator=gen).bfloat16()
    v = torch.randn(n, 1, 256, generator=gen).bfloat16()
    q[:, :, 0] = 1.0
    k[infinite, :, 0] = float("-inf")
    meta = SimpleNamespace(
        query_start_loc=torch.tensor([0, n], dtype=torch.int32, device=DEV),
        seq_lens=torch.tensor([n], dtype=torch.int32, device=DEV),
        counts=torch.tensor([1, n], dtype=torch.int32, device=DEV),
        max_num_reqs=1, max_query_len=n)
    layout = CacheLayout(768, config=OscarConfig(sink_tokens=4, recent_tokens=64))
    out = torch.full((n, 6 * 256), float("nan"), dtype=torch.bfloat16, device=DEV)
    lse = torch.full((n * 6,), float("nan"), dtype=torch.float32, device=DEV)
    kernels.prefill_attention(q.to(DEV), k.to(DEV), v.to(DEV), None, meta, layout, 1 / 16, out,
                              lse)
    torch.cuda.synchronize()
    got = out.cpu().double().view(n, 6, 256)
    got_l = lse.cpu().double().view(n, 6)
    causal = torch.ones(n, n, dtype=torch.bool).tril()
    finite = torch.ones(n, dtype=torch.bool)
    finite[infinite] = False
    seen = causal & finite[None]
    kf = k.double()[:, 0].masked_fill(~finite[:, None], 0.0)
    for h in range(6):
        s = (q.double()[:, h] @ kf.T / 16).masked_fill(~seen, float("-inf"))
        want_l = torch.logsumexp(s, dim=1)
        rows = seen.any(1)
        want = torch.softmax(s[rows], dim=1) @ v.double()[:, 0]
        assert not got[~rows, h].any() and torch.isneginf(got_l[~rows, h]).all()
        assert torch.isfinite(got[:, h]).all()
        assert (got[rows, h] - want).norm() <= 1e-2 * want.norm()
        assert ((got_l[rows, h] - want_l[rows]).abs() <= 2e-2).all()
