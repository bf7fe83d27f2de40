"""Few-row projections whose workgroups own any number of weight rows (``csrc/stream_linear.h``): sizes on either side of every change of that number's
tile and of the rounds, results that start at any address, against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(255, 72), (256, 64), (257, 64), (700, 2088), (4095, 64), (4097, 72), (8191, 64), (8193, 2056), (8195, 2056), (12287, 64), (12289, 72),
                                 (16383, 64), (16385, 64), (32769, 40), (4240, 2048)])
def test_rows_of_a_workgroup(M, N, K):
    from llmctl.ops._lib import native_hybrid

    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    b = torch.randn(N, device="cuda", generator=g).bfloat16()
    want = x.double() @ w.double().t() + b.double()
    got = native_hybrid().rows_linear(x, w, b, 0, N, True)
    assert (got.double() - want).norm() <= 1e-5 * want.norm()  # fp32 sums of K bf16 products: K ulp at most, far less in practice
    assert ((got.double() - want).abs() <= 1e-3).all()  # every output, the edges of the workgroups among them
    assert torch.equal(native_hybrid().rows_linear(x, w, b, 0, N, False), got.bfloat16())


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(255, 512), (257, 520), (700, 504), (4095, 520), (4097, 512), (5119, 504), (5120, 504), (5123, 504), (6143, 2056), (6145, 3072), (8191, 3080), (8193, 520),
                                 (12287, 1024), (12289, 1024), (12289, 1032), (16383, 1024), (16385, 520), (24577, 504), (24577, 520), (8193, 8192), (12289, 8192), (16384, 8192)])
def test_rows_by_the_depth_of_a_sum(M, N, K):
    """Whole tiles below a depth of 512, other numbers of rows from there on, and half as many where rows of W crowd the same channels or are short."""
    test_rows_of_a_workgroup(M, N, K)
