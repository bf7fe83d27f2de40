"""The chunk plans of the scans, on the host: they need no GPU."""

import pytest
import torch

from llmctl.ops import hybrid as hops


@pytest.mark.parametrize("device", ["cpu", torch.device("cpu")])
def test_plans_on_the_host(device):
    cu = [0, 300, 301, 429]
    rows, base, *_, P = hops.gla_chunk_plan(cu, device)
    assert rows.tolist() == [0, 64, 128, 192, 256, 300, 301, 365, 429] and base.tolist() == [0, 5, 6, 8] and P == 8
    rows, seq, base = hops.mlstm_chunk_plan(cu, device, 4, 64, 64)
    assert rows.tolist() == [0, 64, 128, 192, 256, 300, 301, 365, 429] and seq.tolist() == [0] * 5 + [1] + [2] * 2 and base.tolist() == [0, 5, 6, 8]
    assert rows.dtype == torch.int32 and rows.device.type == "cpu"
