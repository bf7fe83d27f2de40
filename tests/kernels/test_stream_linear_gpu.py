"""Few-row projections (``csrc/stream_linear.h``) against float64: row counts at the edges of the row tiles and of the launch rule,
outputs that are no multiple of 4, 16 or 64, K tails, strided rows, bias, activations on some of the columns; and the split of
an unrotated QKV row into q and the paged cache."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _act(name, y):
    F = torch.nn.functional
    return {None: lambda v: v, "gelu": F.gelu, "gelu_tanh": lambda v: F.gelu(v, approximate="tanh"), "relu2": lambda v: torch.relu(v).square()}[name](y)


@pytest.mark.parametrize("M", [1, 2, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(3, 8), (17, 40), (64, 768), (200, 2056), (5119, 96), (5120, 64), (6150, 136), (24570, 72), (24600, 200), (2048, 4096)])
def test_rows_linear_against_float64(M, N, K):
    from llmctl.ops._lib import native, native_hybrid

    g = torch.Generator(device="cuda").manual_seed(M * 7 + N)
    x = torch.randn(M, K + 16, device="cuda", generator=g).bfloat16()[:, 8:8 + K]  # strided rows, 16-byte aligned
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    b = torch.randn(N, device="cuda", generator=g).bfloat16()
    y = x.double() @ w.double().t() + b.double()
    cols = N // 2 + 1
    for act, code in ((None, 0), ("gelu", 1), ("relu2", 3)):
        want = torch.cat([_act(act, y[:, :cols]), y[:, cols:]], 1)
        got = native_hybrid().rows_linear(x, w, b, code, cols, True)
        # fp32 sums of K bf16 products and an fp32 activation: K ulp at most, far less in practice
        assert (got.double() - want).norm() <= 1e-5 * want.norm()
        half = native_hybrid().rows_linear(x, w, b, code, cols, False)
        assert torch.equal(half, got.bfloat16())  # bf16 results are the fp32 ones, rounded once
    want = _act("gelu_tanh", x.double() @ w.double().t())
    got = native().stream_linear(x, w, None, 2)
    assert (got.double() - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("T,nq,nkv,D", [(1, 12, 12, 64), (5, 4, 2, 64), (33, 3, 1, 128)])
def test_qkv_split_cache(T, nq, nkv, D, dtype):
    from llmctl import ops

    g = torch.Generator(device="cuda").manual_seed(T)
    qkv = torch.randn(T, (nq + 2 * nkv) * D, device="cuda", generator=g).bfloat16()
    x = qkv.clone().view(T, nq + 2 * nkv, D)
    caches = [torch.zeros(6, 16, nkv, D, device="cuda").to(dtype) for _ in range(4)]
    slots = torch.randperm(96, device="cuda", generator=g)[:T]
    slots[T // 2] = -1
    q, k, v = ops.qkv_split_cache(qkv, nq, nkv, caches[0], caches[1], slots)
    assert torch.equal(qkv.view_as(x), x)  # the rows are only read
    ops.kv_cache_write(x[:, nq:nq + nkv].contiguous(), x[:, nq + nkv:].contiguous(), caches[2], caches[3], slots)
    assert torch.equal(q, x[:, :nq]) and q.is_contiguous()
    assert torch.equal(k, x[:, nq:nq + nkv]) and torch.equal(v, x[:, nq + nkv:])
    for a, b in ((0, 2), (1, 3)):
        assert torch.equal(caches[a].view(torch.uint8), caches[b].view(torch.uint8))


@pytest.mark.parametrize("M,N,K", [(4, 1040, 6144), (4, 1040, 6272), (5, 2048, 8192), (16, 1024, 6144), (8, 3072, 4224), (16, 8192, 256), (16, 8208, 256),
                                   (8, 8200, 256), (16, 16400, 128), (12, 40976, 128), (6, 50257, 64), (4, 3072, 768), (3, 17, 40), (17, 768, 896),
                                   (12, 2048, 768), (5, 4112, 768), (5, 1024, 1024), (4, 4096, 1536), (4, 4112, 1536), (24, 4096, 1536), (24, 4096, 1664),
                                   (16, 61440, 64), (16, 61424, 64), (8, 4096, 8192), (4, 4096, 8192), (4, 4096, 12288), (8, 4096, 12288), (20, 4240, 1152), (32, 5120, 2048), (24, 2048, 2176), (32, 8208, 128), (33, 64, 128), (8, 64, 20)])
def test_every_form_of_a_few_row_product(M, N, K):
    """The products on either side of every line of the rules, contiguous and strided, with bias and activation, against float64."""
    from llmctl import ops
    from llmctl.ops import hybrid as hops

    g = torch.Generator(device="cuda").manual_seed(M + N)
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    b = torch.randn(N, device="cuda", generator=g).bfloat16()
    wide = torch.randn(M, K + 16, device="cuda", generator=g).bfloat16()
    for x in (wide[:, 8:8 + K].contiguous(), wide[:, 8:8 + K], wide[:, 1:1 + K]):
        y = x.double() @ w.double().t()
        near = lambda got, want: (got.double() - want).norm() <= 2.0 ** -8 * want.norm()  # one rounding of fp32 sums (two with an activation pass)
        assert near(ops.decode_linear(x, w), y) and near(ops.decode_linear(x, w, b), y + b.double())
        if x.data_ptr() % 16 == 0 or M * N % 8 == 0:  # (an activation pass takes multiples of 8)
            assert near(ops.decode_linear(x, w, b, act="gelu"), _act("gelu_tanh", y + b.double()))
        assert near(hops.linear(x, w), y) and near(hops.linear(x, w, b), y + b.double())
        assert (hops.linear_f32(x, w).double() - y).norm() <= 1e-5 * y.norm()
