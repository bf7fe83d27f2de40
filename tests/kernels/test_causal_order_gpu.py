"""The order of causal attention's blocks (``causal_block``): every (head, block) once, whatever the heads of an XCD and the size of a group."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# 8 * n (batch, head) pairs: n heads an XCD in groups of 3 MB of rows, the last group short; ragged last blocks; both head sizes
@pytest.mark.parametrize("B,H,S,D", [(5, 8, 1664, 128), (8, 3, 1000, 64), (4, 2, 200, 128), (1, 8, 129, 64), (3, 24, 256, 64)])
def test_every_block_runs_once(native_lib, B, H, S, D):
    """Outputs and gradients against float32: probabilities and results rounded to bf16 (2^-9 each) and sums of them, 2^-7 of the norm."""
    from llmctl import ops

    g = torch.Generator(device="cuda").manual_seed(S)
    q, k, v, do = (torch.randn(B, S, H, D, generator=g, device="cuda").bfloat16() for _ in range(4))
    leaf = [t.clone().requires_grad_() for t in (q, k, v)]
    o = ops.flash_attention(*leaf, causal=True)
    o.backward(do)
    hide = torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1)
    for b in range(B):
        x = [t[b].float().transpose(0, 1).contiguous().requires_grad_() for t in (q, k, v)]
        p = torch.softmax((x[0] @ x[1].transpose(1, 2).contiguous() / D ** 0.5).masked_fill(hide, float("-inf")), -1)
        want = p @ x[2]
        want.backward(do[b].float().transpose(0, 1))
        for got, ref in [(o[b], want)] + [(t.grad[b], y.grad) for t, y in zip(leaf, x)]:
            e = (got.float().transpose(0, 1) - ref).flatten(1).norm(dim=1)
            assert (e <= 2.0 ** -7 * ref.flatten(1).norm(dim=1)).all()
