"""The small routing kernels at the sizes and values where they can go wrong:
whole and partial waves of experts, ties, signed zeros, masked (-inf) and
infinite logits, against the oracle."""

import pytest
import torch

from flaggems_sglang.ops import fused_moe as fm
from oracle import moe_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scoring", ["softmax", "sigmoid"])
@pytest.mark.parametrize("E", [1, 2, 63, 64, 65, 128, 250, 512, 1023, 1024])
def test_gating_ranks(gpu, E, scoring):
    k = min(E, 64)
    g = torch.Generator().manual_seed(E)
    logits = torch.randn(9, E, generator=g)
    logits[1] = torch.randint(-2, 3, (E,), generator=g).float()      # ties
    logits[2] = torch.where(torch.arange(E) % 2 == 0, 0.0, -0.0)     # equal zeros
    logits[3, : E // 2] = float("-inf")                              # masked experts
    logits[4] = -torch.rand(E, generator=g) * 1e-40                  # denormal, negative
    logits[5] = 80.0 * torch.randn(E, generator=g)                   # scores at 0 and 1
    logits[6, E - 1] = logits[6].max()                               # a tie across the row
    logits[7] = logits[7].bfloat16().float()
    w, ids = fm.fused_topk(torch.empty(9, 8, device=gpu), logits.to(gpu), k, renormalize=False,
                           scoring_func=scoring)
    rw, rids = moe_ref.topk_gating(logits, k, scoring=scoring, renormalize=False)
    assert torch.equal(ids.cpu(), rids)
    # a score: the exponential's and the sum's fp32 rounding (2 ulps each)
    assert torch.allclose(w.cpu(), rw, rtol=2e-6, atol=1e-7)
