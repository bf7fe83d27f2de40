"""The end of the clip norm in one kernel against the same tensor operations: same bits, and the skip rule."""

import pytest
import torch

from llmctl import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsq", [0.0, 1e-30, 0.25, 1.0, 3.0e7, float("inf"), float("nan"), -1.0])
@pytest.mark.parametrize("divisor,limit", [(1.0, 1.0), (3.0, 0.7), (8.0, 0.0), (1.0, 1e9)])
def test_clip_scale(nsq, divisor, limit):
    t, skipped = torch.tensor([nsq], device="cuda"), torch.tensor(4, dtype=torch.int32, device="cuda")
    norm, coef, count = ops.clip_scale(t, skipped, divisor, limit)
    want = torch.sqrt(t) / divisor
    scale = (torch.clamp(limit / (want + 1e-6), max=1.0) if limit else torch.ones_like(want)) / divisor
    scale = torch.where(torch.isfinite(want), scale, torch.full_like(scale, float("nan")))
    assert torch.equal(norm.view(torch.int32), want.view(torch.int32)) or (norm.isnan().all() and want.isnan().all())
    assert torch.equal(coef, scale) or (coef.isnan().all() and scale.isnan().all())
    assert count.shape == () and int(count) == 4 + (not torch.isfinite(want).item()) and int(skipped) == 4
